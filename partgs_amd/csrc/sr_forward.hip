// Forward kernels of the surfel rasteriser for gfx950 (CDNA4, wave64).
//
//   k_preprocess   per surfel: near test, ray-splat homography T, camera-facing
//                  normal, screen AABB and radius, SH -> RGB, and the per-tile
//                  instance histogram (one atomic per covered tile).
//   k_scan_tiles   one workgroup: exclusive scan of the tile histogram into
//                  tile start offsets, tile ranges and the instance count.
//   k_scatter      per surfel: writes a 64-bit key (depth bits << 32 | surfel
//                  id) for every covered tile into that tile's bucket.
//   k_sort_tiles   one workgroup per tile of up to 2048 instances: sorts its
//                  bucket in LDS (depth bins, ranks within a bin), emits
//                  point_list, then splits the sorted list into
//                  per-8x8-quadrant sub-lists.
//   k_split_large  larger tiles cut by depth into segments, which k_sort_tiles
//                  sorts too; k_segment_lists joins their sub-lists.
//   k_blend_fwd    one wave64 per 8 x 8 quadrant, one lane per pixel: front-
//                  to-back alpha blending of colour, depth, alpha, normal,
//                  median depth and depth distortion over the sub-list.
//
// Sorting each tile bucket by (depth bits, surfel id) gives exactly the order
// of the reference's stable radix sort over (tile, depth) keys emitted in
// surfel order (dsr/cuda_rasterizer/rasterizer_impl.cu:70-111, 301-309).
#include <algorithm>

#include "sr_device.h"
#include "sr_internal.h"
#include "sr_pair.h"

namespace sr {

__global__ void k_fill_u32(uint32_t* p, uint32_t v, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

__global__ void k_fill_f32(float* p, float v, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

static unsigned fill_blocks(size_t n) {
  size_t b = (n + 255) / 256;
  if (b > 4096) b = 4096;
  if (b == 0) b = 1;
  return (unsigned)b;
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u32, dim3(fill_blocks(n)), dim3(256), 0, s, p, v, n);
  return hipGetLastError();
}

hipError_t launch_fill_f32(float* p, float v, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_f32, dim3(fill_blocks(n)), dim3(256), 0, s, p, v, n);
  return hipGetLastError();
}

struct F3 {
  float x, y, z;
};
SR_DEV F3 f3(float x, float y, float z) { return F3{x, y, z}; }
SR_DEV F3 operator+(F3 a, F3 b) { return f3(a.x + b.x, a.y + b.y, a.z + b.z); }
SR_DEV F3 operator-(F3 a, F3 b) { return f3(a.x - b.x, a.y - b.y, a.z - b.z); }
SR_DEV F3 operator*(float s, F3 a) { return f3(s * a.x, s * a.y, s * a.z); }

// SH -> RGB, dsr/cuda_rasterizer/forward.cu:20-71 (same association); S(k)
// is coefficient k.
template <typename Get>
SR_DEV F3 color_from_sh_core(int deg, Get S, F3 dir, uint8_t* clamped) {
  F3 res = kSH_C0 * S(0);
  if (deg > 0) {
    const float x = dir.x, y = dir.y, z = dir.z;
    res = res - (kSH_C1 * y) * S(1);
    res = res + (kSH_C1 * z) * S(2);
    res = res - (kSH_C1 * x) * S(3);
    if (deg > 1) {
      const float xx = x * x, yy = y * y, zz = z * z;
      const float xy = x * y, yz = y * z, xz = x * z;
      res = res + (kSH_C2_0 * xy) * S(4);
      res = res + (kSH_C2_1 * yz) * S(5);
      res = res + (kSH_C2_2 * ((2.0f * zz - xx) - yy)) * S(6);
      res = res + (kSH_C2_3 * xz) * S(7);
      res = res + (kSH_C2_4 * (xx - yy)) * S(8);
      if (deg > 2) {
        res = res + ((kSH_C3_0 * y) * (3.0f * xx - yy)) * S(9);
        res = res + ((kSH_C3_1 * xy) * z) * S(10);
        res = res + ((kSH_C3_2 * y) * ((4.0f * zz - xx) - yy)) * S(11);
        res = res + ((kSH_C3_3 * z) * ((2.0f * zz - 3.0f * xx) - 3.0f * yy)) * S(12);
        res = res + ((kSH_C3_4 * x) * ((4.0f * zz - xx) - yy)) * S(13);
        res = res + ((kSH_C3_5 * z) * (xx - yy)) * S(14);
        res = res + ((kSH_C3_6 * x) * (xx - 3.0f * yy)) * S(15);
      }
    }
  }
  res = f3(res.x + 0.5f, res.y + 0.5f, res.z + 0.5f);
  clamped[0] = res.x < 0.0f;
  clamped[1] = res.y < 0.0f;
  clamped[2] = res.z < 0.0f;
  return f3(fmax_(res.x, 0.0f), fmax_(res.y, 0.0f), fmax_(res.z, 0.0f));
}

// Degree 3 over 16 coefficients in a 16-byte aligned row: the row is read as
// twelve float4 (a quarter of the load instructions); otherwise only the
// coefficients the degree uses are read, one float at a time.
SR_DEV F3 color_from_sh(int deg, int M, const float* sh, F3 dir, uint8_t* clamped) {
  if (deg == 3 && M == 16 && (reinterpret_cast<uintptr_t>(sh) & 15u) == 0u) {
    float v[48];
    const float4* s4 = reinterpret_cast<const float4*>(sh);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      const float4 t = s4[i];
      v[4 * i] = t.x;
      v[4 * i + 1] = t.y;
      v[4 * i + 2] = t.z;
      v[4 * i + 3] = t.w;
    }
    return color_from_sh_core(deg, [&](int k) { return f3(v[3 * k], v[3 * k + 1], v[3 * k + 2]); }, dir, clamped);
  }
  return color_from_sh_core(deg, [&](int k) { return f3(sh[3 * k], sh[3 * k + 1], sh[3 * k + 2]); }, dir, clamped);
}

// Screen cull box of a surfel: every pixel where the blend can reach
// alpha >= 1/255 lies inside it.  With rho_max = 2 ln(255 opacity), a pixel
// contributes only if rho3d <= rho_max or rho2d = 2|pix - mean2D|^2 <= rho_max
// (alpha = min(0.99, opacity exp(-rho/2)), dsr/cuda_rasterizer/forward.cu:371-381).
// The box is the union of the disk rho2d <= rho_reject and the bounding box
// of the projected level set rho3d <= rho_reject (the compute_aabb conic with
// cutoff^2 = rho_reject, forward.cu:119-145), where rho_reject exceeds
// rho_max by 0.1% + 0.02, far above FP32 rounding of any pixel's rho.  The
// bounds are on pixel-centre coordinates; pixel i has its centre at
// i + shift (0 here, 0.5 in the _part variant), so the box holds the pixels
// whose centres lie between the bounds.  A level set reaching the camera
// plane (d >= 0) projects unbounded: no box then.
//
// The conic is formed about the surfel's projected centre (ox, oy) = (Tu.z,
// Tv.z) / Tw.z, which lies inside it, so its extents do not cancel against the
// image coordinates: they are good to about 1e-6 of the coordinates.  (mean2D
// would not do: it is the centre of the 3 sigma conic's box, anywhere on or far
// off the image when that conic nearly reaches the camera plane while the
// level set of a faint surfel does not.)  The pixels' own FP32 rho is as good while
// the two planes of a pixel are not nearly parallel (p.z well above the
// rounding of its two products; checked at the centre) and the depth varies
// by less than half over the level set.  Such surfels, nearly all, get a
// margin of 0.02 pixel + 0.2% of the extent + 2e-6 of the coordinate.  The
// others (grazing or very close ones) keep a wide one, with the conic in
// image coordinates, 0.05 pixel + 1e-3 of its coordinates and the bounds
// rounded outwards.  At 300k surfels, 800 x 600, giving the wide margin and
// the outward rounding to all had the acceptance pass evaluate 17.1M box
// pixels for 5.4M accepted pairs; now 8.5M, the pass 107 -> 80 us and the
// per-pair gradient pass, whose chunks are fuller, 107 -> 98 us.
SR_DEV short4 cull_box(F3 Tu, F3 Tv, F3 Tw, float mx, float my, float opa, int W, int H, float shift,
                       float& rho_rej) {
  const short4 none = make_short4(32767, 32767, -32768, -32768);
  const short4 all = make_short4(-32768, -32768, 32767, 32767);
  if (!(opa >= 1.0f / 255.0f)) {
    rho_rej = -1.0f;
    return none;
  }
  const float rho_max = 2.0f * logf(255.0f * opa);
  rho_rej = rho_max * 1.001f + 0.02f;
  const float r2 = sqrtf(0.5f * rho_rej);
  const float c2 = rho_rej;
  const float ww = Tw.x * Tw.x + Tw.y * Tw.y;
  const float d = c2 * ww - Tw.z * Tw.z;
  if (!(d < -1e-3f * (Tw.z * Tw.z))) return all;
  const float fx = c2 / d, fz = -1.0f / d;
  float x0, x1, y0, y1;
  const float ox = Tu.z / Tw.z, oy = Tv.z / Tw.z;
  const F3 U = f3(Tu.x - ox * Tw.x, Tu.y - ox * Tw.y, Tu.z - ox * Tw.z);
  const F3 V = f3(Tv.x - oy * Tw.x, Tv.y - oy * Tw.y, Tv.z - oy * Tw.z);
  const float pa = U.x * V.y, pb = U.y * V.x;
  const bool sound = fabsf(pa - pb) > 0.01f * (fabsf(pa) + fabsf(pb)) && c2 * ww < 0.25f * (Tw.z * Tw.z);
  if (sound) {
    const float cx = fx * (U.x * Tw.x + U.y * Tw.y) + fz * (U.z * Tw.z);
    const float cy = fx * (V.x * Tw.x + V.y * Tw.y) + fz * (V.z * Tw.z);
    const float hx = sqrtf(fmax_(0.0f, cx * cx - (fx * (U.x * U.x + U.y * U.y) + fz * (U.z * U.z))));
    const float hy = sqrtf(fmax_(0.0f, cy * cy - (fx * (V.x * V.x + V.y * V.y) + fz * (V.z * V.z))));
    const float gx = 0.02f + 2e-6f * fmax_(fabsf(mx), fabsf(ox)), gy = 0.02f + 2e-6f * fmax_(fabsf(my), fabsf(oy));
    x0 = ceilf(fmin_(mx - r2, ox - (1.002f * hx - cx)) - gx - shift);
    x1 = floorf(fmax_(mx + r2, ox + (1.002f * hx + cx)) + gx - shift);
    y0 = ceilf(fmin_(my - r2, oy - (1.002f * hy - cy)) - gy - shift);
    y1 = floorf(fmax_(my + r2, oy + (1.002f * hy + cy)) + gy - shift);
  } else {
    const float cx = fx * (Tu.x * Tw.x + Tu.y * Tw.y) + fz * (Tu.z * Tw.z);
    const float cy = fx * (Tv.x * Tw.x + Tv.y * Tw.y) + fz * (Tv.z * Tw.z);
    const float hx = sqrtf(fmax_(0.0f, cx * cx - (fx * (Tu.x * Tu.x + Tu.y * Tu.y) + fz * (Tu.z * Tu.z))));
    const float hy = sqrtf(fmax_(0.0f, cy * cy - (fx * (Tv.x * Tv.x + Tv.y * Tv.y) + fz * (Tv.z * Tv.z))));
    const float mgx = 0.05f + 1e-3f * (fabsf(cx) + hx), mgy = 0.05f + 1e-3f * (fabsf(cy) + hy);
    x0 = floorf(fmin_(mx - r2, cx - hx - mgx) - shift);
    x1 = ceilf(fmax_(mx + r2, cx + hx + mgx) - shift);
    y0 = floorf(fmin_(my - r2, cy - hy - mgy) - shift);
    y1 = ceilf(fmax_(my + r2, cy + hy + mgy) - shift);
  }
  if (!(x0 == x0 && x1 == x1 && y0 == y0 && y1 == y1)) return all;  // NaN: no culling
  x0 = fmax_(x0, -1.0f);
  y0 = fmax_(y0, -1.0f);
  x1 = fmin_(x1, (float)W);
  y1 = fmin_(y1, (float)H);
  if (x1 < x0 || y1 < y0) return none;
  return make_short4((short)x0, (short)y0, (short)x1, (short)y1);
}

// Ray-splat homography and view-space normal of surfel idx seen from view
// v, evaluated in precision R (dsr/cuda_rasterizer/forward.cu:75-115,
// 183-207): T = [L0, 0; L1, 0; p, 1]^T world2ndc ndc2pix, rows Tu, Tv, Tw.
// With R = float the expressions and their order are the reference mode's.
template <typename R> struct Geo {
  R Tu[3], Tv[3], Tw[3], n[3];
};
SR_DEV float sqrt_r(float x) { return sqrtf(x); }
SR_DEV double sqrt_r(double x) { return ::sqrt(x); }
template <typename R>
SR_DEV void surfel_geom(const PreprocessArgs& a, int idx, const float* vm, const float* pm, int W, int H,
                        Geo<R>& g) {
  const R m0 = (R)a.means3D[3 * idx], m1 = (R)a.means3D[3 * idx + 1], m2 = (R)a.means3D[3 * idx + 2];
  if (a.tprec == nullptr) {
    const float* q = a.rots + 4 * idx;
    const R q0 = (R)q[0], q1 = (R)q[1], q2 = (R)q[2], q3 = (R)q[3];
    const R n2 = ((q3 * q3 + q0 * q0) + q1 * q1) + q2 * q2;
    const R s = (R)1 / sqrt_r(n2);
    const R w = q0 * s, x = q1 * s, y = q2 * s, z = q3 * s;
    const R c0[3] = {(R)1 - (R)2 * (y * y + z * z), (R)2 * (x * y + w * z), (R)2 * (x * z - w * y)};
    const R c1[3] = {(R)2 * (x * y - w * z), (R)1 - (R)2 * (x * x + z * z), (R)2 * (y * z + w * x)};
    const R c2[3] = {(R)2 * (x * z + w * y), (R)2 * (y * z - w * x), (R)1 - (R)2 * (x * x + y * y)};
    const R sx = (R)(a.mod * a.scales[2 * idx]), sy = (R)(a.mod * a.scales[2 * idx + 1]);
    const R L0[3] = {sx * c0[0], sx * c0[1], sx * c0[2]};
    const R L1[3] = {sy * c1[0], sy * c1[1], sy * c1[2]};
    auto rowdot = [&](const R* v, int cc) {
      return (v[0] * (R)pm[cc] + v[1] * (R)pm[4 + cc]) + v[2] * (R)pm[8 + cc];
    };
    const R a00 = rowdot(L0, 0), a01 = rowdot(L0, 1), a03 = rowdot(L0, 3);
    const R a10 = rowdot(L1, 0), a11 = rowdot(L1, 1), a13 = rowdot(L1, 3);
    const R pc[3] = {m0, m1, m2};
    const R a20 = rowdot(pc, 0) + (R)pm[12], a21 = rowdot(pc, 1) + (R)pm[13], a23 = rowdot(pc, 3) + (R)pm[15];
    const R hw = (R)W / (R)2, hw1 = (R)(W - 1) / (R)2;
    const R hh = (R)H / (R)2, hh1 = (R)(H - 1) / (R)2;
    g.Tu[0] = a00 * hw + a03 * hw1; g.Tu[1] = a10 * hw + a13 * hw1; g.Tu[2] = a20 * hw + a23 * hw1;
    g.Tv[0] = a01 * hh + a03 * hh1; g.Tv[1] = a11 * hh + a13 * hh1; g.Tv[2] = a21 * hh + a23 * hh1;
    g.Tw[0] = a03; g.Tw[1] = a13; g.Tw[2] = a23;
    for (int i = 0; i < 3; ++i)
      g.n[i] = ((R)vm[i] * c2[0] + (R)vm[4 + i] * c2[1]) + (R)vm[8 + i] * c2[2];
  } else {
    const float* t = a.tprec + 9 * idx;
    for (int i = 0; i < 3; ++i) {
      g.Tu[i] = (R)t[i];
      g.Tv[i] = (R)t[3 + i];
      g.Tw[i] = (R)t[6 + i];
    }
    g.n[0] = (R)0; g.n[1] = (R)0; g.n[2] = (R)1;
  }
}

// compute_aabb with cutoff 3 (dsr/cuda_rasterizer/forward.cu:119-145) up
// to the square roots: the denominator d, the centre p and h0 = p^2 - f T T.
template <typename R> struct Box {
  R d, px, py, h0x, h0y;
};
template <typename R> SR_DEV Box<R> aabb_terms(const Geo<R>& g) {
  Box<R> b;
  const R* Tu = g.Tu;
  const R* Tv = g.Tv;
  const R* Tw = g.Tw;
  b.d = ((R)9 * (Tw[0] * Tw[0]) + (R)9 * (Tw[1] * Tw[1])) + (R)-1 * (Tw[2] * Tw[2]);
  const R inv = (R)1 / b.d;
  const R fx = inv * (R)9, fy = inv * (R)9, fz = inv * (R)-1;
  b.px = (fx * (Tu[0] * Tw[0]) + fy * (Tu[1] * Tw[1])) + fz * (Tu[2] * Tw[2]);
  b.py = (fx * (Tv[0] * Tw[0]) + fy * (Tv[1] * Tw[1])) + fz * (Tv[2] * Tw[2]);
  b.h0x = b.px * b.px - ((fx * (Tu[0] * Tu[0]) + fy * (Tu[1] * Tu[1])) + fz * (Tu[2] * Tu[2]));
  b.h0y = b.py * b.py - ((fx * (Tv[0] * Tv[0]) + fy * (Tv[1] * Tv[1])) + fz * (Tv[2] * Tv[2]));
  return b;
}

// Radius from h0 as the reference forms it, ceil(max(sqrt(max(1e-4, h0x)),
// sqrt(max(1e-4, h0y)), 3 * 0.707106)) (forward.cu:141, 230), in FP32.
SR_DEV int radius_f32(float h0x, float h0y) {
  const float hx = sqrtf(fmax_(1e-4f, h0x));
  const float hy = sqrtf(fmax_(1e-4f, h0y));
  return f2i(ceilf(fmax_(fmax_(hx, hy), 3.0f * kFilterSize)));
}

// The same radius from FP64 h0, exactly: the least integer r >= 3 with
// r^2 >= h0 (the square roots and the ceiling decided on exact squares).
SR_DEV int radius_f64(double h0x, double h0y) {
  const double h0 = fmax(h0x, h0y);
  if (!(h0 < 1.0e18)) return h0 == h0 ? 1000000000 : 3;  // beyond every grid; NaN as the FP32 path's f2i
  int r = (int)ceil(sqrt(fmax(h0, 9.0)));
  while (r > 3 && (double)(r - 1) * (double)(r - 1) >= h0) --r;
  while ((double)r * (double)r < h0) ++r;
  return r;
}

// Near-degenerate surfels, whose FP32 preprocess can take a different
// discrete decision than exact arithmetic would (all tests in FP32 on the
// FP32 values, so the oracle reproduces the selection bit for bit):
//   grazing: |cos| <= 2^-16 (|vx| + |vy| + |vz|), the camera-facing sign
//            test (forward.cu:209-214) within the rounding error of the
//            product and of the unit normal itself, cos == 0 included;
//   conic:   |d| <= 2^-16 (9 Tw.x^2 + 9 Tw.y^2 + Tw.z^2), the AABB
//            denominator (forward.cu:125-126) near its d == 0 exit;
//   tiny:    every tangent entry of Tu, Tv below 2^-7 |Tw.z|, a footprint
//            under 1/128 pixel, where h0 is all cancellation;
//   radius:  h0x or h0y within 2^-20 of its magnitude terms of a square
//            k^2 (k >= 3) where ceil(sqrt(.)) steps (forward.cu:141, 230);
//   edge:    the tile rectangle (getRect, auxiliary.h:67-77) changes when
//            the centre moves by 2^-18 (|p| + 16) pixels.
constexpr float kDegTol = 1.0f / 65536.0f;
SR_DEV bool radius_ambiguous(float h0, float mag) {
  const float e = mag * (1.0f / 1048576.0f);
  const float lo = sqrtf(fmax_(1e-4f, h0 - e)), hi = sqrtf(fmax_(1e-4f, h0 + e));
  return ceilf(fmax_(lo, 3.0f * kFilterSize)) != ceilf(fmax_(hi, 3.0f * kFilterSize));
}
SR_DEV bool rect_ambiguous(float px, float py, int r, int B, int gx, int gy) {
  const float ex = (fabsf(px) + 16.0f) * (1.0f / 262144.0f), ey = (fabsf(py) + 16.0f) * (1.0f / 262144.0f);
  int a0, a1, a2, a3, b0, b1, b2, b3;
  get_rect(px - ex, py - ey, r, B, gx, gy, a0, a1, a2, a3);
  get_rect(px + ex, py + ey, r, B, gx, gy, b0, b1, b2, b3);
  return a0 != b0 || a1 != b1 || a2 != b2 || a3 != b3;
}
SR_DEV bool degenerate(const Geo<float>& g, float vx, float vy, float vz, float cosv, const Box<float>& b, int B,
                       int gx, int gy) {
  const float cabs = (fabsf(vx) + fabsf(vy)) + fabsf(vz);  // |n| = 1; bounds the normal's own error too
  if (!(fabsf(cosv) > kDegTol * cabs)) return true;
  const float dabs = (9.0f * (g.Tw[0] * g.Tw[0]) + 9.0f * (g.Tw[1] * g.Tw[1])) + g.Tw[2] * g.Tw[2];
  if (!(fabsf(b.d) > kDegTol * dabs)) return true;
  const float tmax = fmax_(fmax_(fabsf(g.Tu[0]), fabsf(g.Tu[1])), fmax_(fabsf(g.Tv[0]), fabsf(g.Tv[1])));
  if (tmax < (1.0f / 128.0f) * fabsf(g.Tw[2])) return true;
  const float inv = 1.0f / b.d;
  const float fx = fabsf(inv * 9.0f), fz = fabsf(inv);
  const float mx = b.px * b.px + ((fx * (g.Tu[0] * g.Tu[0]) + fx * (g.Tu[1] * g.Tu[1])) + fz * (g.Tu[2] * g.Tu[2]));
  const float my = b.py * b.py + ((fx * (g.Tv[0] * g.Tv[0]) + fx * (g.Tv[1] * g.Tv[1])) + fz * (g.Tv[2] * g.Tv[2]));
  if (radius_ambiguous(b.h0x, mx) || radius_ambiguous(b.h0y, my)) return true;
  return rect_ambiguous(b.px, b.py, radius_f32(b.h0x, b.h0y), B, gx, gy);
}

// The _part variant's homography, normal and AABB (submodules/
// diff-surfel-rasterization_part, "dsp/": cuda_rasterizer/forward.cu:75-163,
// 235-239): T built in camera space with intrinsics (fx, fy, W/2, H/2), no
// scale modifier, AABB with t = (1, 1, -1), radius ceil(3 max(extent,
// FilterSize)) with the reference's double FilterSize.  Returns false for a
// culled surfel.
constexpr double kPartFS = 0.7071067811865476;
SR_DEV bool part_geom(const PreprocessArgs& a, int idx, const float* vm, const ViewInfo& vi, float vx, float vy,
                      float vz, F3& Tu, F3& Tv, F3& Tw, F3& nrm, float& px, float& py, int& ir) {
  const float fx = (float)vi.W / (2.0f * vi.tanx), fy = (float)vi.H / (2.0f * vi.tany);
  const float cx = (float)((double)(float)vi.W / 2.0), cy = (float)((double)(float)vi.H / 2.0);
  auto Wv = [&](F3 v) {
    return f3((vm[0] * v.x + vm[4] * v.y) + vm[8] * v.z, (vm[1] * v.x + vm[5] * v.y) + vm[9] * v.z,
              (vm[2] * v.x + vm[6] * v.y) + vm[10] * v.z);
  };
  if (a.tprec == nullptr) {
    const float* q = a.rots + 4 * idx;
    const float q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
    const float n2 = ((q3 * q3 + q0 * q0) + q1 * q1) + q2 * q2;
    const float s = 1.0f / sqrtf(n2);
    const float w = q0 * s, x = q1 * s, y = q2 * s, z = q3 * s;
    const F3 c0 = f3(1.0f - 2.0f * (y * y + z * z), 2.0f * (x * y + w * z), 2.0f * (x * z - w * y));
    const F3 c1 = f3(2.0f * (x * y - w * z), 1.0f - 2.0f * (x * x + z * z), 2.0f * (y * z + w * x));
    const F3 c2 = f3(2.0f * (x * z + w * y), 2.0f * (y * z - w * x), 1.0f - 2.0f * (x * x + y * y));
    const float sx = a.scales[2 * idx], sy = a.scales[2 * idx + 1];
    const F3 M0 = Wv(sx * c0), M1 = Wv(sy * c1);
    F3 tn = Wv(c2);
    const float cosv = ((-tn.x * vx) + (-tn.y * vy)) + (-tn.z * vz);
    if (cosv == 0.0f) return false;  // BACKFACE_CULL
    tn = (cosv > 0.0f ? 1.0f : -1.0f) * tn;
    Tu = f3(fx * M0.x + cx * M0.z, fx * M1.x + cx * M1.z, fx * vx + cx * vz);
    Tv = f3(fy * M0.y + cy * M0.z, fy * M1.y + cy * M1.z, fy * vy + cy * vz);
    Tw = f3(M0.z, M1.z, vz);
    nrm = tn;
  } else {
    const float* t = a.tprec + 9 * idx;
    Tu = f3(t[0], t[1], t[2]);
    Tv = f3(t[3], t[4], t[5]);
    Tw = f3(t[6], t[7], t[8]);
    nrm = f3(0.0f, 0.0f, 1.0f);  // left unset by the reference
  }
  const float d = (1.0f * (Tw.x * Tw.x) + 1.0f * (Tw.y * Tw.y)) + -1.0f * (Tw.z * Tw.z);
  if (d == 0.0f) return false;
  const float inv = 1.0f / d;
  const float f0 = 1.0f * inv, f1 = 1.0f * inv, f2 = -1.0f * inv;
  px = (f0 * (Tu.x * Tw.x) + f1 * (Tu.y * Tw.y)) + f2 * (Tu.z * Tw.z);
  py = (f0 * (Tv.x * Tw.x) + f1 * (Tv.y * Tw.y)) + f2 * (Tv.z * Tw.z);
  const float h0x = px * px - ((f0 * (Tu.x * Tu.x) + f1 * (Tu.y * Tu.y)) + f2 * (Tu.z * Tu.z));
  const float h0y = py * py - ((f0 * (Tv.x * Tv.x) + f1 * (Tv.y * Tv.y)) + f2 * (Tv.z * Tv.z));
  const float hx = sqrtf(fmax_(0.0f, h0x)), hy = sqrtf(fmax_(0.0f, h0y));
  const float radius = (float)ceil(3.0 * fmax((double)fmaxf(hx, hy), kPartFS));
  ir = f2i(radius);
  return true;
}

// Forward preprocess of surfel idx in view v (record r = v * P + idx),
// dsr/cuda_rasterizer/forward.cu:75-145, 148-251.  Returns false for culled
// surfels, else its tile rectangle in the view's tile grid.  Near-degenerate
// surfels (see degenerate()) take the homography, normal, camera-facing
// test and AABB in FP64 and store them rounded to FP32.
SR_DEV bool preprocess_one(const PreprocessArgs& a, int v, int idx, size_t r, int& x0, int& y0, int& x1,
                           int& y1) {
  a.radii[r] = 0;
  a.tiles[r] = 0;
  const float m0 = a.means3D[3 * idx], m1 = a.means3D[3 * idx + 1], m2 = a.means3D[3 * idx + 2];
  const float* vm = a.vm + 16 * v;
  const float* pm = a.pm + 16 * v;
  const float* campos = a.campos + 3 * v;
  const int W = a.vs.v[v].W, H = a.vs.v[v].H, gx = a.vs.v[v].gx, gy = a.vs.v[v].gy;
  const float vx = ((vm[0] * m0 + vm[4] * m1) + vm[8] * m2) + vm[12];
  const float vy = ((vm[1] * m0 + vm[5] * m1) + vm[9] * m2) + vm[13];
  const float vz = ((vm[2] * m0 + vm[6] * m1) + vm[10] * m2) + vm[14];
  if (vz <= 0.2f) {
    if (a.prefiltered) atomicOr(&a.counters[1], kErrPrefiltered);
    return false;
  }
  F3 Tu, Tv, Tw, nrm;
  float px, py, mult;
  int ir;
  if (a.part) {
    if (!part_geom(a, idx, vm, a.vs.v[v], vx, vy, vz, Tu, Tv, Tw, nrm, px, py, ir)) return false;
    mult = 1.0f;
  } else {
  Geo<float> g;
  surfel_geom<float>(a, idx, vm, pm, W, H, g);
  const float cosv = -((vx * g.n[0] + vy * g.n[1]) + vz * g.n[2]);
  Box<float> b = aabb_terms(g);
  if (!degenerate(g, vx, vy, vz, cosv, b, a.vs.B, gx, gy)) {
    mult = cosv > 0.0f ? 1.0f : -1.0f;
    Tu = f3(g.Tu[0], g.Tu[1], g.Tu[2]);
    Tv = f3(g.Tv[0], g.Tv[1], g.Tv[2]);
    Tw = f3(g.Tw[0], g.Tw[1], g.Tw[2]);
    nrm = mult * f3(g.n[0], g.n[1], g.n[2]);
    px = b.px;
    py = b.py;
    ir = radius_f32(b.h0x, b.h0y);
  } else {
    Geo<double> G;
    surfel_geom<double>(a, idx, vm, pm, W, H, G);
    const double dvx = (((double)vm[0] * m0 + (double)vm[4] * m1) + (double)vm[8] * m2) + (double)vm[12];
    const double dvy = (((double)vm[1] * m0 + (double)vm[5] * m1) + (double)vm[9] * m2) + (double)vm[13];
    const double dvz = (((double)vm[2] * m0 + (double)vm[6] * m1) + (double)vm[10] * m2) + (double)vm[14];
    const double dcos = -((dvx * G.n[0] + dvy * G.n[1]) + dvz * G.n[2]);
    if (dcos == 0.0) return false;
    const Box<double> B = aabb_terms(G);
    if (B.d == 0.0) return false;
    mult = dcos > 0.0 ? 1.0f : -1.0f;
    Tu = f3((float)G.Tu[0], (float)G.Tu[1], (float)G.Tu[2]);
    Tv = f3((float)G.Tv[0], (float)G.Tv[1], (float)G.Tv[2]);
    Tw = f3((float)G.Tw[0], (float)G.Tw[1], (float)G.Tw[2]);
    nrm = mult * f3((float)G.n[0], (float)G.n[1], (float)G.n[2]);
    px = (float)B.px;
    py = (float)B.py;
    ir = radius_f64(B.h0x, B.h0y);
    mult *= 2.0f;  // marks the record as evaluated in FP64
  }
  }
  // the rectangle from the stored (FP32) centre, as the scatter recomputes it
  get_rect(px, py, ir, a.vs.B, gx, gy, x0, y0, x1, y1);
  const uint32_t area = (uint32_t)(x1 - x0) * (uint32_t)(y1 - y0);
  if (area == 0) return false;
  F3 rgb;
  if (a.colors == nullptr) {
    const F3 dir0 = f3(m0 - campos[0], m1 - campos[1], m2 - campos[2]);
    const float len = sqrtf((dir0.x * dir0.x + dir0.y * dir0.y) + dir0.z * dir0.z);
    const F3 dir = f3(dir0.x / len, dir0.y / len, dir0.z / len);
    uint8_t cl[3];
    rgb = color_from_sh(a.D, a.M, a.shs + (size_t)idx * a.M * 3, dir, cl);
    uchar4 c4;
    c4.x = cl[0];
    c4.y = cl[1];
    c4.z = cl[2];
    c4.w = 0;
    reinterpret_cast<uchar4*>(a.clamped)[r] = c4;
  } else {
    rgb = f3(a.colors[3 * idx], a.colors[3 * idx + 1], a.colors[3 * idx + 2]);
  }
  const float opa = a.opac[idx];
  float rho_rej;
  const short4 box = cull_box(Tu, Tv, Tw, px, py, opa, W, H, a.part ? 0.5f : 0.0f, rho_rej);
  a.depths[r] = vz;
  a.radii[r] = ir;
  float4* rc = a.rec + (size_t)kRecQuads * r;
  rc[0] = make_float4(Tu.x, Tu.y, Tu.z, Tv.x);
  rc[1] = make_float4(Tv.y, Tv.z, Tw.x, Tw.y);
  rc[2] = make_float4(Tw.z, px, py, opa);
  rc[3] = make_float4(nrm.x, nrm.y, nrm.z, rgb.x);
  rc[4] = make_float4(rgb.y, rgb.z, rho_rej, mult);
  a.cullbox[r] = box;
  a.tiles[r] = area;
  return true;
}

// Tile histograms with up to kHistTiles tiles are gathered in LDS per
// workgroup and flushed with one global atomic per non-empty bin, which
// keeps hot tiles (thousands of instances) off a single global counter.
constexpr int kHistTiles = 4096;

// Exclusive scan of one value per lane over a group of 256 consecutive lanes
// (four waves; a workgroup holds one or more groups, s_w four words each);
// every lane must call it.  Returns the lane's exclusive prefix and the
// group's total.
SR_DEV uint32_t group_scan256(uint32_t x, uint32_t* s_w, uint32_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, first = wave & ~3;
  uint32_t incl = x;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)incl, d);
    if (lane >= d) incl += y;
  }
  if (lane == 63) s_w[wave] = incl;
  __syncthreads();
  uint32_t off = 0;
  for (int w = first; w < wave; ++w) off += s_w[w];
  total = (s_w[first] + s_w[first + 1]) + (s_w[first + 2] + s_w[first + 3]);
  return off + incl - x;
}

// A workgroup per (surfel block, view), so its tile histogram is that view's.
// Each workgroup also stores its records' slot total in ssum (view-major),
// which the tile scan turns into the first slot of every workgroup.  Workgroups
// go to the XCDs in turn: every eighth one takes the next view of the same
// surfels, so that one XCD's L2 holds a block's SHs (48 KB) for all its views:
// 1.03 ms for a million surfels and 16 views, 1.36 with all surfels of a view
// before the next view.
// Partial-gradient slots of a record: one per (instance, quadrant holding
// it), the quadrants found as the sort's sub-lists find them.
SR_DEV uint32_t record_slots(short4 bx, int x0, int y0, int x1, int y1, int B, const ViewInfo& vi) {
  const int QX = B / kQuad;
  return (uint32_t)(quad_span(bx.x, bx.z, x0 * QX, x1 * QX, vi.W) * quad_span(bx.y, bx.w, y0 * QX, y1 * QX, vi.H));
}

constexpr int kXcds = 8;
__global__ __launch_bounds__(256) void k_preprocess(PreprocessArgs a) {
  __shared__ uint32_t s_hist[kHistTiles];
  __shared__ uint32_t s_ssum[4];
  const int blocks = (a.P + 255) / 256;
  const int turn = blockIdx.x / kXcds;
  const int v = turn % a.vs.V, block = turn / a.vs.V * kXcds + blockIdx.x % kXcds;
  if (block >= blocks) return;
  const int gx = a.vs.v[v].gx;
  const int T = gx * a.vs.v[v].gy;
  uint32_t* tile_count = a.tile_count + a.vs.v[v].tile_base;
  const bool lds = T <= kHistTiles;
  if (lds)
    for (int t = threadIdx.x; t < T; t += blockDim.x) s_hist[t] = 0;
  const int idx = block * 256 + threadIdx.x;
  int x0 = 0, y0 = 0, x1 = 0, y1 = 0;
  const bool ok = idx < a.P && preprocess_one(a, v, idx, (size_t)v * a.P + idx, x0, y0, x1, y1);
  {
    uint32_t total = 0;
    // the cull box was stored by preprocess_one (this thread)
    const uint32_t ns = ok ? record_slots(a.cullbox[(size_t)v * a.P + idx], x0, y0, x1, y1, a.vs.B, a.vs.v[v]) : 0u;
    (void)group_scan256(ns, s_ssum, total);
    if (threadIdx.x == 0) a.ssum[(size_t)v * blocks + block] = total;
  }
  if (ok) {
    for (int ty = y0; ty < y1; ++ty)
      for (int tx = x0; tx < x1; ++tx) {
        if (lds) atomicAdd(&s_hist[ty * gx + tx], 1u);
        else atomicAdd(&tile_count[ty * gx + tx], 1u);
      }
  }
  if (lds) {
    __syncthreads();
    for (int t = threadIdx.x; t < T; t += blockDim.x) {
      const uint32_t c = s_hist[t];
      if (c) atomicAdd(&tile_count[t], c);
    }
  }
}

hipError_t launch_preprocess(const PreprocessArgs& a, hipStream_t s) {
  if (a.P == 0 || a.vs.V == 0) return hipSuccess;
  const int blocks = (a.P + 255) / 256;
  hipLaunchKernelGGL(k_preprocess, dim3((blocks + kXcds - 1) / kXcds * kXcds * a.vs.V), dim3(256), 0, s, a);
  return hipGetLastError();
}


// Exclusive scan of N values per lane over a 1024-lane workgroup: each wave
// scans its 64 lanes with shuffles, one wave scans the 16 wave totals, so
// the workgroup meets at three barriers instead of two per doubling step.
// s: 32 N words of LDS.  Returns the lane's exclusive prefixes in x and the
// workgroup totals in total.
template <int N>
SR_DEV void scan1024_excl(uint32_t* s, uint32_t (&x)[N], uint32_t (&total)[N]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t incl[N];
#pragma unroll
  for (int k = 0; k < N; ++k) incl[k] = x[k];
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const uint32_t y = (uint32_t)__shfl_up((int)incl[k], off, 64);
      if (lane >= off) incl[k] += y;
    }
  }
  __syncthreads();  // s may still be read by a previous scan
  if (lane == 63) {
#pragma unroll
    for (int k = 0; k < N; ++k) s[k * 32 + wave] = incl[k];
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      uint32_t t = lane < 16 ? s[k * 32 + lane] : 0u;
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)t, off, 64);
        if (lane >= off) t += y;
      }
      if (lane < 16) s[k * 32 + 16 + lane] = t;  // inclusive over the waves
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t base = wave == 0 ? 0u : s[k * 32 + 16 + wave - 1];
    total[k] = s[k * 32 + 31];
    x[k] = base + incl[k] - x[k];
  }
}

// Exclusive scan of the tile histogram by one 1024-lane workgroup, with the
// list of tiles above kSmallMax instances (count in counters[3]) and the
// number of each one's first kSegKeys-key segment (seg_off, followed by the
// total, which also goes to counters[6]);
// then the same scan for the per-workgroup slot totals of the preprocess (in
// place), which numbers every record's slots in record order.  host (pinned
// memory, may be null) receives what the caller waits for, the instances
// [0], error flags [1] and slots [8]: a copy command after the kernel is a
// launch of its own in the stream.  Without the two of them a forward and
// backward of 300k surfels at 800 x 600 takes 679 us instead of 683.
constexpr int kScanThreads = 1024;
__global__ __launch_bounds__(kScanThreads) void k_scan_tiles(int T, const uint32_t* count,
                                                              uint32_t* start, uint32_t* fill,
                                                              uint32_t* ranges, uint32_t* counters,
                                                              uint32_t capacity, int nb, uint32_t* ssum,
                                                              uint32_t slot_capacity,
                                                              uint32_t* large, uint32_t* seg_off, uint32_t* host) {
  __shared__ uint32_t s_part[3 * 32];
  const int tid = threadIdx.x;
  auto each = [](const uint32_t* x, int b, int e, auto&& fn) {  // eight loads in flight
    int i = b;
    for (; i + 8 <= e; i += 8) {
      uint32_t v[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) v[t] = x[i + t];
#pragma unroll
      for (int t = 0; t < 8; ++t) fn(i + t, v[t]);
    }
    for (; i < e; ++i) fn(i, x[i]);
  };
  const int per = (T + kScanThreads - 1) / kScanThreads;
  const int b = tid * per;
  const int e = min(T, b + per);
  // this lane's tiles: instances, large tiles, their segments
  uint32_t v3[3] = {0u, 0u, 0u}, tot3[3];
  each(count, b, e, [&](int, uint32_t c) {
    v3[0] += c;
    if (c > (uint32_t)kSmallMax) {
      v3[1] += 1u;
      v3[2] += segments_of(c);
    }
  });
  scan1024_excl(s_part, v3, tot3);
  uint32_t run = v3[0], at = v3[1], sat = v3[2];
  each(count, b, e, [&](int i, uint32_t c) {
    start[i] = run;
    fill[i] = run;
    ranges[2 * i] = c ? run : 0u;
    ranges[2 * i + 1] = c ? run + c : 0u;
    run += c;
    if (c > (uint32_t)kSmallMax) {
      large[at] = (uint32_t)i;
      seg_off[at++] = sat;
      sat += segments_of(c);
    }
  });
  if (tid == kScanThreads - 1) {
    start[T] = tot3[0];
    counters[0] = tot3[0];
    if (tot3[0] > capacity) atomicOr(&counters[1], kErrCapacity);
    counters[3] = tot3[1];
    counters[6] = tot3[2];
    seg_off[tot3[1]] = tot3[2];
  }
  // the per-workgroup slot totals of the preprocess, in place
  const int pb = (nb + kScanThreads - 1) / kScanThreads;
  const int b2 = tid * pb, e2 = min(nb, b2 + pb);
  uint32_t w1[1] = {0u}, wt[1];
  each(ssum, b2, e2, [&](int, uint32_t d) { w1[0] += d; });
  scan1024_excl(s_part, w1, wt);
  uint32_t run3 = w1[0];
  each(ssum, b2, e2, [&](int i, uint32_t d) {
    ssum[i] = run3;
    run3 += d;
  });
  if (tid == 0) {
    counters[8] = wt[0];
    if (wt[0] > slot_capacity) atomicOr(&counters[1], kErrCapacity | kErrSlots);
  }
  if (host == nullptr) return;
  __syncthreads();
  if (tid == 0) {
    host[0] = tot3[0];
    host[1] = __hip_atomic_load(&counters[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    host[8] = wt[0];
  }
}

hipError_t launch_scan_tiles(int T, const uint32_t* count, uint32_t* start, uint32_t* fill,
                             uint32_t* ranges, uint32_t* counters, uint32_t capacity, int nb, uint32_t* ssum,
                             uint32_t slot_capacity, uint32_t* large, uint32_t* seg_off, uint32_t* host,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(kScanThreads), 0, s, T, count, start, fill, ranges,
                     counters, capacity, nb, ssum, slot_capacity, large, seg_off, host);
  return hipGetLastError();
}

// duplicateWithKeys, rasterizer_impl.cu:70-111, writing straight into tile
// buckets.  With few enough tiles, each workgroup first counts its instances
// per tile in LDS, reserves one contiguous block per tile with a single
// global atomic, then hands out slots inside the block with LDS atomics.
// The key's low word is the record number, which orders equal depths by
// record exactly as the reference's (tile | depth, record) sort does.  Beside
// each key goes what the sort would otherwise gather per entry from all over
// the records: the instance's first partial-gradient slot and its quadrant
// mask (pay).  Bound by the global atomics on the hot tiles and the chain
// behind them: 1,024 surfels a workgroup make a quarter of the atomics 256 do.
// 300k surfels at 800 x 600: 21 us, where 256 surfels a workgroup and 8-byte
// (record, slot) pairs stored by instance number took 41; a million surfels
// and 16 views: 528 us, was 901.
constexpr int kScatterThreads = 1024;
__global__ __launch_bounds__(kScatterThreads) void k_scatter(ScatterArgs a) {
  __shared__ uint32_t s_cnt[kHistTiles];
  __shared__ uint32_t s_base[kHistTiles];
  __shared__ uint32_t s_ssum[kScatterThreads / 64];
  if (a.counters[1] & kErrCapacity) return;
  const int v = blockIdx.y;
  const int B = a.vs.B, gx = a.vs.v[v].gx, gy = a.vs.v[v].gy;
  const int T = gx * gy;
  uint32_t* tile_fill = a.tile_fill + a.vs.v[v].tile_base;
  const bool lds = T <= kHistTiles;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t r = (size_t)v * a.P + idx;
  int x0 = 0, y0 = 0, x1 = 0, y1 = 0;
  uint64_t key = 0;
  const bool ok = idx < a.P && a.radii[r] > 0;
  if (ok) {
    const float4 q2 = a.rec[(size_t)kRecQuads * r + 2];
    get_rect(q2.y, q2.z, a.radii[r], B, gx, gy, x0, y0, x1, y1);
    key = (uint64_t)__float_as_uint(a.depths[r]) << 32 | (uint32_t)r;
  }
  // partial-gradient slots: the record's run, and each instance's first
  // slot (its quadrants' slots follow in quadrant order)
  const ViewInfo& vi = a.vs.v[v];
  const short4 bx = ok ? a.cullbox[r] : make_short4(32767, 32767, -32768, -32768);
  const uint32_t ns = ok ? record_slots(bx, x0, y0, x1, y1, B, vi) : 0u;
  const int groups = (a.P + 255) / 256;  // of 256 records, per view, as the preprocess counted them
  const int group = min(idx / 256, groups - 1);
  uint32_t total = 0;
  const uint32_t slot0 = a.ssum[(size_t)v * groups + group] + group_scan256(ns, s_ssum, total);
  if (idx < a.P) a.rslot[r] = make_uint2(slot0, ns);
  const int QX = B / kQuad;
  // quadrant columns and rows of the image that the box meets
  const int qc0 = bx.x > 0 ? bx.x / kQuad : 0, qc1 = min(bx.z >= 0 ? bx.z / kQuad : -1, (vi.W - 1) / kQuad);
  const int qr0 = bx.y > 0 ? bx.y / kQuad : 0, qr1 = min(bx.w >= 0 ? bx.w / kQuad : -1, (vi.H - 1) / kQuad);
  // place(t) gives the bucket position of this lane's instance in tile t
  auto emit = [&](auto&& place) {
    uint32_t sl = slot0;
    for (int ty = y0; ty < y1; ++ty) {
      const int ra = max(qr0 - ty * QX, 0), rb = min(qr1 - ty * QX, QX - 1);
      for (int tx = x0; tx < x1; ++tx) {
        const int ca = max(qc0 - tx * QX, 0), cb = min(qc1 - tx * QX, QX - 1);
        const uint32_t cols = ca <= cb ? (2u << cb) - (1u << ca) : 0u;
        uint32_t mask = 0u;
        for (int q = ra; q <= rb; ++q) mask |= cols << (q * QX);
        const uint32_t at = place(ty * gx + tx);
        a.keys[at] = key;
        a.pay[at] = make_uint2(sl, mask);
        sl += (uint32_t)__popc(mask);
      }
    }
  };
  if (!lds) {
    if (ok) emit([&](int t) { return atomicAdd(&tile_fill[t], 1u); });
    return;
  }
  for (int t = threadIdx.x; t < T; t += blockDim.x) s_cnt[t] = 0;
  __syncthreads();
  if (ok)
    for (int ty = y0; ty < y1; ++ty)
      for (int tx = x0; tx < x1; ++tx) atomicAdd(&s_cnt[ty * gx + tx], 1u);
  __syncthreads();
  for (int t = threadIdx.x; t < T; t += blockDim.x) {
    const uint32_t c = s_cnt[t];
    if (c) s_base[t] = atomicAdd(&tile_fill[t], c);
    s_cnt[t] = 0;
  }
  __syncthreads();
  if (ok) emit([&](int t) { return s_base[t] + atomicAdd(&s_cnt[t], 1u); });
}

hipError_t launch_scatter(const ScatterArgs& a, hipStream_t s) {
  if (a.P == 0 || a.vs.V == 0) return hipSuccess;
  hipLaunchKernelGGL(k_scatter, dim3((a.P + kScatterThreads - 1) / kScatterThreads, a.vs.V), dim3(kScatterThreads), 0,
                     s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Per-tile sort.  A tile of up to kSmallMax instances is sorted in LDS by one
// 512-lane workgroup.  A larger one is first split by depth into segments of
// about kSegKeys keys (k_split_large), which are then sorted like small tiles.
// ---------------------------------------------------------------------------

// LDS slot of key i in the merge sort: one pad slot after every K keys, so
// the K-strided accesses of a wave (lane t at t K + k) spread over the banks
// instead of piling onto two of them.
template <int K>
SR_DEV int lds_slot(int i) {
  return i + i / K;
}

// Ascending sort of S keys in LDS by NT lanes, K keys per lane (S a power
// of two, K <= S <= NT K; key i at lds_slot(i)).  Each lane sorts its run of
// K in registers with a bitonic network, then log2(S / K) merge-path levels
// double the sorted runs: at each level a lane finds, by binary search,
// where its K outputs start in the two runs it merges and merges them in
// registers.  A level costs a lane about log2(S) + K dependent LDS reads,
// against the S / NT compare-exchange sweeps per step of an LDS bitonic
// sort.  Keys must be unique apart from the ~0 padding.
template <int NT, int K>
SR_DEV void merge_sort_lds(uint64_t* v, int S) {
  const int tid = threadIdx.x;
  const bool act = tid * K < S;
  auto at = [&](int i) -> uint64_t { return v[lds_slot<K>(i)]; };
  uint64_t r[K];
  if (act) {
#pragma unroll
    for (int k = 0; k < K; ++k) r[k] = at(tid * K + k);
#pragma unroll
    for (int kk = 2; kk <= K; kk <<= 1) {
#pragma unroll
      for (int j = kk >> 1; j > 0; j >>= 1) {
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int l = i ^ j;
          if (l > i) {
            const uint64_t x = r[i], y = r[l];
            if (((i & kk) == 0) ? (x > y) : (x < y)) {
              r[i] = y;
              r[l] = x;
            }
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) v[lds_slot<K>(tid * K + k)] = r[k];  // the lane's own slots: no hazard
  }
  __syncthreads();
  for (int w = K; w < S; w <<= 1) {
    if (act) {
      const int o = tid * K;
      const int g = o & ~(2 * w - 1);  // first key of the two runs this lane merges
      const int kq = o - g;
      // co-rank: how many of the first kq merged keys come from run A
      // (ties from B, matching the merge below)
      int lo = max(0, kq - w), hi = min(kq, w);
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (at(g + mid) < at(g + w + kq - mid - 1)) lo = mid + 1;
        else hi = mid;
      }
      int i = lo, j = kq - lo;
      uint64_t av = i < w ? at(g + i) : ~0ull, bv = j < w ? at(g + w + j) : ~0ull;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const bool ta = av < bv;  // ties (padding only) from B
        r[k] = ta ? av : bv;
        if (ta) {
          ++i;
          av = i < w ? at(g + i) : ~0ull;
        } else {
          ++j;
          bv = j < w ? at(g + w + j) : ~0ull;
        }
      }
    }
    __syncthreads();
    if (act) {
#pragma unroll
      for (int k = 0; k < K; ++k) v[lds_slot<K>(tid * K + k)] = r[k];
    }
    __syncthreads();
  }
}

SR_DEV int next_pow2(int n) {
  int s = 1;
  while (s < n) s <<= 1;
  return s;
}

// Quadrant sub-lists.  Sub-list q of tile t is the tile's sorted list with
// the entries removed whose conservative cull box misses quadrant q (such
// an entry cannot reach alpha >= 1/255 anywhere in the quadrant, so blending
// the sub-list gives the reference's result); it starts at Q * beg + q * n
// and holds (surfel id, position in the tile list) pairs.  Each non-empty
// sub-list appends its 64-entry chunks to the acceptance work list.

// Called by one whole wave; lane q < Q holds the length of the tile's
// sub-list q.  Writes the lengths and clears the overflow flags, and appends
// the sub-lists' 64-entry chunks to the acceptance work list with one atomic
// for the tile (same-address atomics serialise).
SR_DEV void append_work(const SortArgs& a, int tile, int Q, uint32_t cnt) {
  const int lane = threadIdx.x & 63;
  const bool has = lane < Q;
  const uint32_t nch = has ? (cnt + 63u) / 64u : 0u;
  uint32_t incl = nch;
#pragma unroll
  for (int d = 1; d < kMaxQuads; d <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)incl, d);
    if (lane >= d) incl += y;
  }
  const uint32_t all = (uint32_t)__shfl((int)incl, kMaxQuads - 1);
  uint32_t w0 = 0;
  if (lane == 0 && all > 0) w0 = atomicAdd(a.work_count, all);
  w0 = (uint32_t)__shfl((int)w0, 0);
  if (has) {
    const uint32_t qi = (uint32_t)(tile * Q + lane);
    a.sub_count[qi] = cnt;
    a.q_flag[qi] = 0u;
    const uint32_t first = w0 + incl - nch;
    const int B = a.vs.B, QX = B / kQuad;
    const uint32_t view = (uint32_t)view_of_tile(a.vs, (uint32_t)tile);
    const int lt = tile - (int)a.vs.v[view].tile_base, gx = a.vs.v[view].gx;
    const int x0 = lt % gx * B + lane % QX * kQuad, y0 = lt / gx * B + lane / QX * kQuad;
    const uint32_t beg = a.ranges[2 * tile], n = a.ranges[2 * tile + 1] - beg;
    const size_t e0 = (size_t)Q * beg + (size_t)lane * n;
    for (uint32_t ch = 0; ch < nch; ++ch)
      a.work[first + ch] = pack_work(qi, e0 + 64u * ch, min(64u, cnt - 64u * ch), view, x0, y0);
  }
}

// LDS of a tile sort: K keys per lane of NT, and NB bins.
template <int NT, int K, int NB> struct TileLds {
  static constexpr int kKeys = NT * K;
  // the keys (the merge sort pads them by one slot per K), then the bins
  static constexpr int kBytes = (kKeys + NT) * 8 > kKeys * 8 + (NB + 1) * 4 ? (kKeys + NT) * 8 : kKeys * 8 + (NB + 1) * 4;
};

// Keys whose depths share one bin are ranked against each other, so a tile
// with a fuller bin than this (equal or nearly equal depths) goes through the
// merge sort instead.
constexpr uint32_t kBinMax = 128;

// Sorts the n <= NT K keys of a bucket at `src` and returns in ent[r], for
// sorted entry r NT + tid, the record (the key's low word) and the entry's
// place in the unsorted bucket.
//
// The depths are cut into NB equal bins between the tile's smallest and
// largest (depth bits, a monotone map), the keys counted into the bins, the
// bins scanned, and the keys placed by bin; a key's rank is then its bin's
// start plus the number of smaller keys in the bin.  Keys are unique, so this
// is the sorted order whatever order the lanes arrive in.  About 6 + n / NB
// dependent LDS accesses a key, where the merge sort it falls back to makes 50
// to 300.
template <int NT, int K, int NB>
SR_DEV void sort_bucket(const uint64_t* src, int n, char* lds, uint2 (&ent)[K]) {
  constexpr int NW = NT / 64, per = NB / NT;
  static_assert(NB % NT == 0, "whole bins per lane");
  __shared__ uint32_t s_w[NW];
  __shared__ uint32_t s_red[2][NW];
  __shared__ uint32_t s_full;
  uint64_t* keys = reinterpret_cast<uint64_t*>(lds);
  uint32_t* bins = reinterpret_cast<uint32_t*>(lds + (size_t)NT * K * 8);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // all K loads in flight: unconditional, the index clamped into the bucket
  uint64_t kv[K];
#pragma unroll
  for (int r = 0; r < K; ++r) kv[r] = src[min(r * NT + tid, n - 1)];
  uint32_t lo = 0xFFFFFFFFu, hi = 0u;
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const uint32_t d = (uint32_t)(kv[r] >> 32);
    lo = min(lo, d);
    hi = max(hi, d);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, off, 64));
    hi = max(hi, (uint32_t)__shfl_xor((int)hi, off, 64));
  }
  if (lane == 0) {
    s_red[0][wave] = lo;
    s_red[1][wave] = hi;
  }
  if (tid == 0) s_full = 0u;
#pragma unroll
  for (int t = 0; t < per; ++t) bins[t * NT + tid] = 0u;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    lo = min(lo, s_red[0][w]);
    hi = max(hi, s_red[1][w]);
  }
  const float scale = (float)NB / ((float)(hi - lo) + 1.0f);
  auto bin_of = [&](uint64_t k) {
    return min(NB - 1, (int)((float)((uint32_t)(k >> 32) - lo) * scale));
  };
  uint32_t at[K];
#pragma unroll
  for (int r = 0; r < K; ++r)
    if (r * NT + tid < n) at[r] = atomicAdd(&bins[bin_of(kv[r])], 1u);
  __syncthreads();
  uint32_t c[per], sum = 0u, top = 0u;
#pragma unroll
  for (int t = 0; t < per; ++t) {
    c[t] = bins[tid * per + t];
    sum += c[t];
    top = max(top, c[t]);
  }
  uint32_t incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)incl, off, 64);
    if (lane >= off) incl += y;
  }
  if (lane == 63) s_w[wave] = incl;
  if (top > kBinMax) s_full = 1u;
  __syncthreads();
  if (s_full != 0u) {  // uniform
#pragma unroll
    for (int r = 0; r < K; ++r) keys[lds_slot<K>(r * NT + tid)] = r * NT + tid < n ? kv[r] : ~0ull;
    __syncthreads();
    merge_sort_lds<NT, K>(keys, max(next_pow2(n), K));
    // each lane's own keys' ranks: lower bounds in the sorted keys
#pragma unroll
    for (int r = 0; r < K; ++r) {
      uint32_t below = 0u;
      for (int w = NT * K / 2; w > 0; w >>= 1)
        if ((int)below + w <= n && keys[lds_slot<K>((int)below + w - 1)] < kv[r]) below += (uint32_t)w;
      at[r] = below;
    }
  } else {
    uint32_t run = incl - sum;
#pragma unroll
    for (int w = 0; w < NW; ++w) run += w < wave ? s_w[w] : 0u;
#pragma unroll
    for (int t = 0; t < per; ++t) {
      bins[tid * per + t] = run;
      run += c[t];
    }
    if (tid == NT - 1) bins[NB] = run;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < K; ++r)
      if (r * NT + tid < n) keys[bins[bin_of(kv[r])] + at[r]] = kv[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < K; ++r) {
      at[r] = 0u;
      if (r * NT + tid < n) {
        const int b = bin_of(kv[r]);
        const uint32_t b0 = bins[b], b1 = bins[b + 1];
        uint32_t below = b0;
        for (uint32_t m = b0; m < b1; ++m) below += keys[m] < kv[r] ? 1u : 0u;
        at[r] = below;
      }
    }
  }
  __syncthreads();
  uint2* order = reinterpret_cast<uint2*>(lds);
#pragma unroll
  for (int r = 0; r < K; ++r)
    if (r * NT + tid < n) order[at[r]] = make_uint2((uint32_t)kv[r], (uint32_t)(r * NT + tid));
  __syncthreads();
#pragma unroll
  for (int r = 0; r < K; ++r) ent[r] = order[min(r * NT + tid, n - 1)];
  __syncthreads();
}

// Writes point_list, first slot and quadrant mask of the cnt sorted entries
// from tile-list position pos on (entry r NT + tid: record ent[r].x, payload
// pay[ent[r].y]), consecutive lanes at consecutive positions, and returns the
// masks (none past the end).
template <int NT, int K>
SR_DEV void place_entries(const SortArgs& a, const uint2* pay, uint32_t pos, int cnt, const uint2 (&ent)[K],
                          uint32_t (&hm)[K]) {
  const int tid = threadIdx.x;
  uint2 p[K];  // all loads in flight
#pragma unroll
  for (int r = 0; r < K; ++r) p[r] = pay[ent[r].y];
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const int i = r * NT + tid;
    hm[r] = i < cnt ? p[r].y : 0u;
    if (i < cnt) {
      a.point_list[pos + i] = ent[r].x;
      a.pos_slot[pos + i] = p[r].x;
      a.pos_quads[pos + i] = (uint16_t)hm[r];
    }
  }
}

// Appends entries r NT + tid (record rid[r], quadrants hm[r], position
// first + r NT + tid in the tile's list) to the tile's quadrant sub-lists in
// order.  Per quadrant, the hits of every (round, wave) are counted by ballot
// and scanned by one wave.  s_base[q]: entries the sub-list holds already;
// advanced by the new ones.
template <int NT, int K>
SR_DEV void append_sublists(const SortArgs& a, uint32_t beg, int n, int first, int Q, const uint32_t (&rid)[K],
                            const uint32_t (&hm)[K], uint32_t* s_cnt, uint32_t* s_base) {
  constexpr int NW = NT / 64, E = K * NW;  // counts per quadrant, in entry order
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int r = 0; r < K; ++r) {
    for (int q = 0; q < Q; ++q) {  // uniform
      const uint64_t m = __ballot((hm[r] >> q) & 1u);
      if (lane == 0) s_cnt[q * E + r * NW + wave] = (uint32_t)__popcll(m);
    }
  }
  __syncthreads();
  for (int q = wave; q < Q; q += NW) {
    static_assert(E <= 64, "one count a lane");
    const uint32_t c = lane < E ? s_cnt[q * E + lane] : 0u;
    uint32_t incl = c;
#pragma unroll
    for (int off = 1; off < E; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)incl, off, 64);
      if (lane >= off) incl += y;
    }
    const uint32_t b0 = s_base[q];
    if (lane < E) s_cnt[q * E + lane] = b0 + incl - c;
    if (lane == E - 1) s_base[q] = b0 + incl;
  }
  __syncthreads();
  uint2* base = a.sub + (size_t)Q * beg;
  const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
  for (int r = 0; r < K; ++r) {
    for (int q = 0; q < Q; ++q) {
      const bool hit = (hm[r] >> q) & 1u;
      const uint64_t m = __ballot(hit);
      if (hit)
        base[(size_t)q * n + s_cnt[q * E + r * NW + wave] + (uint32_t)__popcll(m & lt)] =
            make_uint2(rid[r], (uint32_t)(first + r * NT + tid));
    }
  }
  __syncthreads();  // the counts are rewritten by the next call
}

// Number of elements of A among the first k of merge(A, B) (keys unique).
SR_DEV int co_rank(const uint64_t* A, int na, const uint64_t* Bv, int nb, int k) {
  int lo = max(0, k - nb), hi = min(k, na);
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (A[mid] < Bv[k - mid - 1]) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// The large tiles' split, one 1024-lane workgroup per tile of the scan's list
// (striding): the depths are cut into kSplitBins equal bins between the tile's
// smallest and largest, and the keys moved bin by bin into key2.  Segment s of
// the tile starts at the first bin boundary at or after kSegKeys s keys, so
// segments hold kSegKeys keys give or take a bin, and their sorts, one
// workgroup each, put the tile in order; the payloads move along, loaded with
// the keys: 20 us for 300k surfels at 800 x 600 and 768 for a million and 16
// views; 24 and 1,153 with each payload's load behind the stores of the one
// before.  A segment above kSmallMax keys (more
// than kSegKeys nearly equal depths in one bin) is sorted here: chunks in LDS,
// then pairwise merges between the tile's two key buffers.
constexpr int kSplitThreads = 1024, kSplitBins = 4096, kSplitRun = 4;
constexpr int kSplitChunk = kSplitThreads * kSplitRun;  // keys of one LDS merge sort

// Sorts n keys at v by chunks and merges; other: a buffer as large.
SR_DEV void sort_range(uint64_t* v, uint64_t* other, int n, uint64_t* lds) {
  constexpr int NT = kSplitThreads, K = kSplitRun;
  const int tid = threadIdx.x;
  for (int c0 = 0; c0 < n; c0 += kSplitChunk) {
    const int cn = min(kSplitChunk, n - c0);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int i = tid + k * NT;
      lds[lds_slot<K>(i)] = i < cn ? v[c0 + i] : ~0ull;
    }
    __syncthreads();
    merge_sort_lds<NT, K>(lds, max(next_pow2(cn), K));
    for (int i = tid; i < cn; i += NT) v[c0 + i] = lds[lds_slot<K>(i)];
  }
  __syncthreads();
  uint64_t *src = v, *dst = other;
  for (int w = kSplitChunk; w < n; w <<= 1) {
    for (int a0 = 0; a0 < n; a0 += 2 * w) {
      const int na = min(w, n - a0), nb = max(0, min(w, n - a0 - w));
      const uint64_t *A = src + a0, *Bv = src + a0 + na;
      uint64_t* out = dst + a0;
      const int total = na + nb, per = (total + NT - 1) / NT;
      const int k0 = min(total, tid * per), k1 = min(total, k0 + per);
      if (k0 < k1) {
        int i = co_rank(A, na, Bv, nb, k0);
        int j = k0 - i;
        for (int k = k0; k < k1; ++k) {
          if (j >= nb || (i < na && A[i] < Bv[j])) out[k] = A[i++];
          else out[k] = Bv[j++];
        }
      }
    }
    __syncthreads();
    uint64_t* t = src;
    src = dst;
    dst = t;
  }
  if (src != v)
    for (int i = tid; i < n; i += NT) v[i] = src[i];
  __syncthreads();
}

__global__ __launch_bounds__(kSplitThreads) void k_split_large(SortArgs a) {
  constexpr int NT = kSplitThreads, NB = kSplitBins, per = NB / NT, kU = 8, NW = NT / 64;
  __shared__ __align__(16) uint64_t lds[kSplitChunk + NT];  // the bins, or a chunk of the fallback
  __shared__ uint32_t s_lo[NW], s_hi[NW], s_w[NW];
  static_assert(sizeof(lds) >= (NB + 1) * 4, "the bins fit");
  if (a.counters[1] & kErrCapacity) return;
  uint32_t* bins = reinterpret_cast<uint32_t*>(lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (uint32_t l = blockIdx.x; l < a.counters[3]; l += gridDim.x) {
    const int tile = (int)a.large[l];
    const uint32_t beg = a.ranges[2 * tile];
    const int n = (int)(a.ranges[2 * tile + 1] - beg);
    const uint64_t* src = a.keys + beg;
    uint64_t* dst = a.key2 + beg;
    uint32_t* seg = a.seg_start + a.seg_off[l];
    const int nseg = (int)segments_of((uint32_t)n);
    auto each = [&](auto&& fn) {  // every key of the tile with its place, kU loads in flight a lane
      for (int i0 = 0; i0 < n; i0 += kU * NT) {
        uint64_t k[kU];
#pragma unroll
        for (int t = 0; t < kU; ++t) k[t] = src[min(i0 + t * NT + tid, n - 1)];
#pragma unroll
        for (int t = 0; t < kU; ++t)
          if (i0 + t * NT + tid < n) fn(k[t], i0 + t * NT + tid);
      }
    };
    uint32_t lo = 0xFFFFFFFFu, hi = 0u;
    each([&](uint64_t k, int) {
      const uint32_t d = (uint32_t)(k >> 32);
      lo = min(lo, d);
      hi = max(hi, d);
    });
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      lo = min(lo, (uint32_t)__shfl_xor((int)lo, off, 64));
      hi = max(hi, (uint32_t)__shfl_xor((int)hi, off, 64));
    }
    __syncthreads();  // the previous tile's readers are done
    if (lane == 0) {
      s_lo[wave] = lo;
      s_hi[wave] = hi;
    }
#pragma unroll
    for (int t = 0; t < per; ++t) bins[t * NT + tid] = 0u;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      lo = min(lo, s_lo[w]);
      hi = max(hi, s_hi[w]);
    }
    const float scale = (float)NB / ((float)(hi - lo) + 1.0f);
    auto bin_of = [&](uint64_t k) { return min(NB - 1, (int)((float)((uint32_t)(k >> 32) - lo) * scale)); };
    each([&](uint64_t k, int) { atomicAdd(&bins[bin_of(k)], 1u); });
    __syncthreads();
    uint32_t c[per], sum = 0u;
#pragma unroll
    for (int t = 0; t < per; ++t) {
      c[t] = bins[tid * per + t];
      sum += c[t];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)incl, off, 64);
      if (lane >= off) incl += y;
    }
    if (lane == 63) s_w[wave] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
#pragma unroll
    for (int w = 0; w < NW; ++w) run += w < wave ? s_w[w] : 0u;
    // segment s starts at the first bin boundary that is >= kSegKeys s
#pragma unroll
    for (int t = 0; t < per; ++t) {
      bins[tid * per + t] = run;
      const uint32_t end = run + c[t];
      for (uint32_t sg = run / kSegKeys + 1u; sg <= end / kSegKeys && sg < (uint32_t)nseg; ++sg) seg[sg] = beg + end;
      run = end;
    }
    if (tid == 0) seg[0] = beg;
    __syncthreads();
    const uint2* pay = a.pay + beg;
    uint2* pay2 = a.pay2 + beg;
    for (int i0 = 0; i0 < n; i0 += kU * NT) {  // keys and payloads in flight together
      uint64_t k[kU];
      uint2 p[kU];
      uint32_t at[kU];
#pragma unroll
      for (int t = 0; t < kU; ++t) {
        const int i = min(i0 + t * NT + tid, n - 1);
        k[t] = src[i];
        p[t] = pay[i];
      }
#pragma unroll
      for (int t = 0; t < kU; ++t) at[t] = i0 + t * NT + tid < n ? atomicAdd(&bins[bin_of(k[t])], 1u) : 0u;
#pragma unroll
      for (int t = 0; t < kU; ++t)
        if (i0 + t * NT + tid < n) {
          dst[at[t]] = k[t];
          pay2[at[t]] = p[t];
        }
    }
    __syncthreads();
    for (int sg = 0; sg < nseg; ++sg) {  // uniform
      const uint32_t s0 = seg[sg], s1 = sg + 1 < nseg ? seg[sg + 1] : beg + (uint32_t)n;
      if (s1 - s0 > (uint32_t)kSmallMax) {
        // merges between key2 and the tile's sub-list space (8 bytes an
        // instance and quadrant, not written yet); the payloads then follow
        // their keys by binary search
        const int Q = quads_per_tile(a.vs.B), m = (int)(s1 - s0);
        uint64_t* v = a.key2 + s0;
        sort_range(v, reinterpret_cast<uint64_t*>(a.sub + (size_t)Q * s0), m, lds);
        const uint64_t first = v[0], last = v[m - 1];
        each([&](uint64_t k, int i) {
          if (k < first || k > last) return;
          int lo2 = 0, hi2 = m - 1;  // v[lo2] <= k
          while (lo2 < hi2) {
            const int mid = (lo2 + hi2 + 1) >> 1;
            if (v[mid] <= k) lo2 = mid;
            else hi2 = mid - 1;
          }
          pay2[(s0 - beg) + (uint32_t)lo2] = pay[i];
        });
        __syncthreads();
      }
    }
  }
}

// Large tile and segment of segment item `it` (< counters[6]).
struct Segment {
  int tile, n, nseg, sg;
  uint32_t beg, s0, item0;  // tile's first key, segment's first, item of segment 0
  int cnt;
};
SR_DEV Segment segment_item(const SortArgs& a, uint32_t it) {
  uint32_t lo = 0, hi = a.counters[3];  // seg_off[lo] <= it < seg_off[hi]
  while (hi - lo > 1u) {
    const uint32_t mid = (lo + hi) >> 1;
    if (a.seg_off[mid] <= it) lo = mid;
    else hi = mid;
  }
  Segment g;
  g.tile = (int)a.large[lo];
  g.beg = a.ranges[2 * g.tile];
  g.n = (int)(a.ranges[2 * g.tile + 1] - g.beg);
  g.nseg = (int)segments_of((uint32_t)g.n);
  g.item0 = a.seg_off[lo];
  g.sg = (int)(it - g.item0);
  g.s0 = a.seg_start[it];
  g.cnt = (int)((g.sg + 1 < g.nseg ? a.seg_start[it + 1] : g.beg + (uint32_t)g.n) - g.s0);
  return g;
}

// Small tiles and segments, one 512-lane workgroup each: the first seg_blocks
// workgroups stride over the segments (workgroups b, b + seg_blocks, ...), so
// these start first; workgroup seg_blocks + t sorts tile t when it holds at
// most kSmallMax instances.  A segment's quadrant hits are counted here and its
// sub-list entries placed by k_segment_lists.  Latency-bound: 300k surfels at
// 800 x 600 put about 1,650 instances in each of 350 tiles, so a CU holds two
// or three sorts and what counts is each one's chain of LDS and gather
// latencies.  25 us there, and 481 for a million surfels and 16 views, where
// looking each entry's record up by instance number and then its cull box took
// 38 and 1,031.  256-lane merge sorts of 8 keys a lane, with larger tiles cut
// into 2,048-key chunks merged by rank (and above 16,384 by one workgroup),
// took 92 us (with the split and the segments' lists now 60) and 624 us for 1M
// surfels at 1237 x 823.  One workgroup for each tile of up to 16,384 was no
// better than those on the tiles it bounds (75 us for 8,192 keys, 132 us for
// 16,384).
constexpr int kSortThreads = 512, kSortKeys = kSmallMax / 512, kSortBins = 2048;
__global__ __launch_bounds__(kSortThreads) void k_sort_tiles(SortArgs a, uint32_t seg_blocks) {
  constexpr int NT = kSortThreads, K = kSortKeys;
  __shared__ __align__(16) char lds[TileLds<NT, K, kSortBins>::kBytes];
  __shared__ uint32_t s_base[kMaxQuads];
  static_assert(kMaxQuads * K * (NT / 64) * 4 <= (int)sizeof(lds), "the quadrant counts fit");
  if (a.counters[1] & kErrCapacity) return;
  const int Q = quads_per_tile(a.vs.B);
  const int tid = threadIdx.x;
  uint2 ent[K];
  uint32_t rid[K], hm[K];
  if (blockIdx.x < seg_blocks) {
    for (uint32_t it = blockIdx.x; it < a.counters[6]; it += seg_blocks) {
      const Segment g = segment_item(a, it);
      if (tid < Q) s_base[tid] = 0u;
      __syncthreads();
      // one round, unless the segment was too full for one and is sorted already
      for (int c0 = 0; c0 < g.cnt; c0 += NT * K) {
        const int cn = min(NT * K, g.cnt - c0);
        if (g.cnt <= NT * K) {
          sort_bucket<NT, K, kSortBins>(a.key2 + g.s0, cn, lds, ent);
        } else {
#pragma unroll
          for (int r = 0; r < K; ++r) {
            const int i = min(r * NT + tid, cn - 1);
            ent[r] = make_uint2((uint32_t)a.key2[g.s0 + c0 + i], (uint32_t)i);
          }
        }
        place_entries<NT, K>(a, a.pay2 + g.s0 + c0, g.s0 + c0, cn, ent, hm);
        for (int q = 0; q < Q; ++q) {
          uint32_t hits = 0;
#pragma unroll
          for (int r = 0; r < K; ++r) hits += (uint32_t)__popcll(__ballot((hm[r] >> q) & 1u));
          if ((tid & 63) == 0 && hits) atomicAdd(&s_base[q], hits);
        }
      }
      __syncthreads();
      if (tid < Q) a.seg_hits[(size_t)it * Q + tid] = s_base[tid];
      __syncthreads();
    }
    return;
  }
  const int tile = (int)(blockIdx.x - seg_blocks);
  const uint32_t beg = a.ranges[2 * tile];
  const int n = (int)(a.ranges[2 * tile + 1] - beg);
  if (n > kSmallMax) return;
  if (n <= 0) {
    if (tid < Q) {
      a.sub_count[(size_t)tile * Q + tid] = 0;
      a.q_flag[(size_t)tile * Q + tid] = 0u;
    }
    return;
  }
  sort_bucket<NT, K, kSortBins>(a.keys + beg, n, lds, ent);
  place_entries<NT, K>(a, a.pay + beg, beg, n, ent, hm);
#pragma unroll
  for (int r = 0; r < K; ++r) rid[r] = ent[r].x;
  if (tid < Q) s_base[tid] = 0u;
  __syncthreads();
  append_sublists<NT, K>(a, beg, n, 0, Q, rid, hm, reinterpret_cast<uint32_t*>(lds), s_base);
  if (tid < 64) append_work(a, tile, Q, tid < Q ? s_base[tid] : 0u);
}

// The segments' sub-list entries, one workgroup each (striding): a segment's
// entries follow those of the tile's earlier segments.  The first segment's
// workgroup also writes the sub-list lengths and the acceptance work items.
__global__ __launch_bounds__(kSortThreads) void k_segment_lists(SortArgs a) {
  constexpr int NT = kSortThreads, K = kSortKeys;
  __shared__ uint32_t s_cnt[kMaxQuads * K * (NT / 64)];
  __shared__ uint32_t s_base[kMaxQuads], s_all[kMaxQuads];
  if (a.counters[1] & kErrCapacity) return;
  const int Q = quads_per_tile(a.vs.B);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (uint32_t it = blockIdx.x; it < a.counters[6]; it += gridDim.x) {
    const Segment g = segment_item(a, it);
    for (int q = wave; q < Q; q += NT / 64) {
      uint32_t before = 0u, all = 0u;
      for (int t = lane; t < g.nseg; t += 64) {
        const uint32_t h = a.seg_hits[(size_t)(g.item0 + (uint32_t)t) * Q + q];
        all += h;
        before += t < g.sg ? h : 0u;
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        before += (uint32_t)__shfl_xor((int)before, off, 64);
        all += (uint32_t)__shfl_xor((int)all, off, 64);
      }
      if (lane == 0) {
        s_base[q] = before;
        s_all[q] = all;
      }
    }
    __syncthreads();
    if (g.sg == 0 && wave == 0) append_work(a, g.tile, Q, lane < Q ? s_all[lane] : 0u);
    for (int c0 = 0; c0 < g.cnt; c0 += NT * K) {
      uint32_t rid[K], hm[K];
#pragma unroll
      for (int r = 0; r < K; ++r) {
        const int i = c0 + r * NT + tid;
        const uint32_t pos = g.s0 + (uint32_t)min(i, g.cnt - 1);
        rid[r] = a.point_list[pos];
        hm[r] = a.pos_quads[pos];
      }
#pragma unroll
      for (int r = 0; r < K; ++r) hm[r] = c0 + r * NT + tid < g.cnt ? hm[r] : 0u;
      append_sublists<NT, K>(a, g.beg, g.n, (int)(g.s0 - g.beg) + c0, Q, rid, hm, s_cnt, s_base);
    }
    __syncthreads();
  }
}

hipError_t launch_sort_tiles(const SortArgs& a, size_t max_segments, hipStream_t s) {
  if (a.vs.T == 0) return hipSuccess;
  const unsigned T = (unsigned)a.vs.T;
  // as many workgroups as run at once several times over, so the uneven
  // tiles and segments of a large batch balance
  const unsigned segs = (unsigned)std::min<size_t>(max_segments, 8192);
  hipLaunchKernelGGL(k_split_large, dim3(std::min(T, 4096u)), dim3(kSplitThreads), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_sort_tiles, dim3(segs + T), dim3(kSortThreads), 0, s, a, segs);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_segment_lists, dim3(segs), dim3(kSortThreads), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Acceptance pass.  One wave per (quadrant, chunk of 64 sub-list entries):
// bit j of pixel p's mask is set when entry j of the chunk reaches
// alpha >= 1/255 at p.  Only pixels inside an entry's cull box can (the box
// holds every such pixel), so the wave evaluates exactly the (entry, pixel)
// pairs of the boxes clipped to the quadrant, 64 pairs per step: SlotOwner
// names the entry of every pair slot, and the slot's offset in the
// entry's box gives the pixel.  The bits go to per-pixel masks in LDS; each
// accepted pair adds -log2(1 - alpha) in 2^-20 to its pixel's sum, from which
// the chunk's transmittance follows.  That transmittance is only compared
// against half the saturation threshold, a margin of a factor 2 against its
// rounding.  LDS atomics bound the pass where they are wide or on floats: with
// a 64-bit or and a float add a pair it took 77 us (299 for 1M surfels at
// 1237 x 823), with two 32-bit integer ones 60 (212); with a byte per pair slot
// naming its entry, whose 4 KB left room for half the waves, 80 (338).  The chunks of all quadrants are independent, so this, the
// bulk of the pair evaluations, runs balanced over the whole GPU; the blend
// kernels then visit only accepted pairs.
// ---------------------------------------------------------------------------
constexpr float kLogUnit = 1048576.0f;  // 64 pairs of alpha <= 0.99 sum to less than 2^29 of it
template <bool kPart>
__global__ __launch_bounds__(64) void k_accept(AcceptArgs a) {
  __shared__ float4 s_q0[64], s_q1[64], s_q2[64];
  __shared__ float s_rej[64];
  __shared__ uint32_t s_start[64];  // running box area before entry j
  __shared__ uint32_t s_geo[64];    // entry j's clipped box: x0 | y0 << 4 | w << 8
  __shared__ uint32_t s_mask[2][64];  // per pixel: entries 0..31 and 32..63
  __shared__ uint32_t s_logT[64];   // per pixel: sum of -log2(1 - alpha) over its accepted pairs, in 2^-20
  __shared__ uint32_t s_head[64];
  // r / w for r < 64 and 1 <= w <= 8 as (r * kDiv[w]) >> 9
  constexpr uint32_t kDiv[9] = {0u, 512u, 256u, 171u, 128u, 103u, 86u, 74u, 64u};
  const int lane = threadIdx.x;
  if (a.counters[1] & kErrCapacity) return;
  const uint32_t nwork = *a.work_count;
  for (uint32_t w = blockIdx.x; w < nwork; w += gridDim.x) {
    const WorkItem it = unpack_work(a.work[nwork - 1u - w]);  // from the end: see work_capacity
    const ViewInfo& vi = a.vs.v[it.view];
    const int qx0 = it.x0, qy0 = it.y0;
    const int qw = min(kQuad, vi.W - qx0), qh = min(kQuad, vi.H - qy0);  // pixels inside the image
    wave_lds_fence();  // the previous item's readers are done
    uint32_t area = 0, geo = 0;
    if ((uint32_t)lane < it.m) {
      const uint32_t rid = a.sub[it.first + lane].x;
      const float4* r = a.rec + (size_t)kRecQuads * rid;
      s_q0[lane] = r[0];
      s_q1[lane] = r[1];
      s_q2[lane] = r[2];
      s_rej[lane] = r[4].z;
      const short4 bx = a.cullbox[rid];
      const int x0 = max((int)bx.x - qx0, 0), x1 = min((int)bx.z - qx0, qw - 1);
      const int y0 = max((int)bx.y - qy0, 0), y1 = min((int)bx.w - qy0, qh - 1);
      if (x1 >= x0 && y1 >= y0) {
        const uint32_t bw = (uint32_t)(x1 - x0 + 1);
        area = bw * (uint32_t)(y1 - y0 + 1);
        geo = (uint32_t)x0 | ((uint32_t)y0 << 4) | (bw << 8);
      }
    }
    uint32_t incl = area;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t v = (uint32_t)__shfl_up((int)incl, off, 64);
      if (lane >= off) incl += v;
    }
    const uint32_t total = (uint32_t)__shfl((int)incl, 63, 64);  // at most 64 boxes of 64 pixels
    const uint32_t first = incl - area;
    s_start[lane] = first;
    s_geo[lane] = geo;
    s_mask[0][lane] = s_mask[1][lane] = 0u;
    s_logT[lane] = 0u;
    wave_lds_fence();
    SlotOwner owner;
    for (uint32_t base = 0; base < total; base += 64) {
      const uint32_t t = base + (uint32_t)lane;
      const int j = (int)owner.at(s_head, base, first, area);
      if (t < total) {
        const uint32_t g = s_geo[j];
        const uint32_t r = t - s_start[j], bw = (g >> 8) & 15u;
        const uint32_t dy = (r * kDiv[bw]) >> 9, dx = r - dy * bw;
        const int lx = (int)(g & 15u) + (int)dx, ly = (int)((g >> 4) & 15u) + (int)dy;
        Pair e;
        if (eval_pair<true>(pixel_centre<kPart>(qx0 + lx), pixel_centre<kPart>(qy0 + ly), s_q0[j], s_q1[j], s_q2[j],
                            s_rej[j], e)) {
          const int p = ly * kQuad + lx;
          atomicOr(&s_mask[j >> 5][p], 1u << (j & 31));
          atomicAdd(&s_logT[p], (uint32_t)(__log2f(1.0f - e.alpha) * -kLogUnit));
        }
      }
    }
    wave_lds_fence();
    const size_t slot = it.first + 64u * (size_t)it.qi + lane;
    a.masks[slot] = (uint64_t)s_mask[1][lane] << 32 | s_mask[0][lane];
    a.chunk_T[slot] = exp2f((float)s_logT[lane] * (-1.0f / kLogUnit));
  }
}

hipError_t launch_accept(const AcceptArgs& a, size_t max_items, hipStream_t s) {
  if (max_items == 0) return hipSuccess;
  const unsigned grid = (unsigned)(max_items < kChunkBlocks ? max_items : kChunkBlocks);
  if (a.part) hipLaunchKernelGGL(k_accept<true>, dim3(grid), dim3(64), 0, s, a);
  else hipLaunchKernelGGL(k_accept<false>, dim3(grid), dim3(64), 0, s, a);
  return hipGetLastError();
}

// Transmittance below which a pixel is certainly saturated.  The blend stops
// a pixel at its first pair with T (1 - alpha) < 1e-4, T the running product
// of (1 - alpha) over its accepted pairs in order.  The chunk transmittances
// give the same product through sums of log2(1 - alpha): with hardware
// log2 / exp2 (relative error near 2^-22 each) that is off by far less than a
// factor 2 even over thousands of pairs, so below half the threshold the
// pixel stopped in an earlier chunk.
constexpr float kSaturatedT = 0.5e-4f;

// Pair-store offsets: one wave per quadrant, one lane per pixel.  Each
// pixel gets one contiguous run of the store for its accepted pairs (in
// entry order, across every chunk), so the per-pixel blend chains read one
// stream; frag_off[chunk, pixel] records where each chunk's pairs begin.
// Chunks behind a pixel's saturation point (by the acceptance pass's chunk
// transmittances) are cut: their masks are cleared and their pairs never
// stored, as the blend never reaches them.  A quadrant whose pairs do not
// fit is flagged and left to the staged path.
// Bound by the chain of loads down the longest lists (hundreds of chunks in a
// dense tile), so lists above kPoChunks chunks are walked by four waves, each
// kPoChunks of every 4 kPoChunks, which exchange their transmittances and
// counts per pixel in LDS; lists that one step covers are read once.  26 us for
// 300k surfels at 800 x 600 and 230 for 16 views of a million, where one wave
// a quadrant took 37 and 363; eight waves: 25 and 259.  Reserving the runs of
// 16 quadrants with one atomic made a workgroup wait for its longest list: 30
// and 530.
constexpr int kPoWaves = 4, kPoChunks = 8;
__global__ __launch_bounds__(kPoWaves * 64) void k_pair_offsets(AcceptArgs a) {
  constexpr int kU = kPoChunks;  // chunks in flight a wave
  __shared__ float s_T[kPoWaves][64];
  __shared__ int s_cut[kPoWaves][64];
  __shared__ uint32_t s_n[kPoWaves][64];
  __shared__ unsigned long long s_fill;
  const int B = a.vs.B, QX = B / kQuad, Q = QX * QX;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (a.counters[1] & kErrCapacity) return;
  const int qi = blockIdx.x;
  const int tile = qi / Q, q = qi % Q;
  const int cnt = (int)a.sub_count[qi];
  const int nch = (cnt + 63) / 64;
  const int nw = nch > kU ? kPoWaves : 1;  // uniform
  if (wave >= nw) return;
  auto sync = [&]() {
    if (nw > 1) __syncthreads();
  };
  const uint32_t rbeg = a.ranges[2 * tile], ntile = a.ranges[2 * tile + 1] - rbeg;
  const size_t base = mask_base(Q, rbeg, ntile, tile, q) + lane;
  const int step = nw * kU;
  uint64_t mk[kU];
  // unconditional loads (chunk index clamped into the list) so all are in
  // flight together; the values past the end are then dropped
  auto load_masks = [&](int c0) {
#pragma unroll
    for (int k = 0; k < kU; ++k) mk[k] = a.masks[base + (size_t)min(c0 + k, nch - 1) * 64];
  };
  uint32_t tot = 0, n = 0;  // the pixel's pairs; of this wave's chunks of the step
  int cut = nch;            // first chunk the pixel cannot reach
  float T0 = 1.0f;          // transmittance in front of the step
  for (int t0 = 0; t0 < nch; t0 += step) {
    const int c0 = t0 + wave * kU;
    load_masks(c0);
    float tk[kU], T = T0, all = 1.0f;
#pragma unroll
    for (int k = 0; k < kU; ++k) tk[k] = a.chunk_T[base + (size_t)min(c0 + k, nch - 1) * 64];
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      tk[k] = c0 + k < nch ? tk[k] : 1.0f;
      all *= tk[k];
    }
    if (nw > 1) {
      s_T[wave][lane] = all;
      __syncthreads();
      all = 1.0f;
#pragma unroll
      for (int w = 0; w < kPoWaves; ++w) {
        if (w == wave) T = T0 * all;
        all *= s_T[w][lane];
      }
    }
    T0 *= all;
    int first = cut;
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      if (T < kSaturatedT) first = min(first, c0 + k);
      T *= tk[k];
    }
    cut = first;
    if (nw > 1) {
      s_cut[wave][lane] = first;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kPoWaves; ++w) cut = min(cut, s_cut[w][lane]);
    }
    n = 0;
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      if (c0 + k >= cut) {
        mk[k] = 0ull;
        if (c0 + k < nch) a.masks[base + (size_t)(c0 + k) * 64] = 0ull;
      }
      n += (uint32_t)__popcll(mk[k]);
    }
    if (nw > 1) {
      s_n[wave][lane] = n;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kPoWaves; ++w) tot += s_n[w][lane];
    } else {
      tot += n;
    }
  }
  uint32_t incl = tot;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t v = __shfl_up(incl, off, 64);
    if (lane >= off) incl += v;
  }
  const uint32_t total = __shfl(incl, 63, 64);
  unsigned long long qbase = 0;
  if (threadIdx.x == 0 && total > 0) qbase = atomicAdd(a.frag_fill, (unsigned long long)total);
  qbase = __shfl(qbase, 0, 64);
  if (nw > 1) {
    if (threadIdx.x == 0) s_fill = qbase;
    __syncthreads();
    qbase = s_fill;
  }
  const bool fits = qbase + total <= (unsigned long long)a.frag_cap;
  if (wave == 0) {
    // cost of the quadrant for the blend kernels' longest-first order: its
    // longest pixel chain (the staged path, when it does not fit, its list)
    uint32_t mx = tot;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = max(mx, (uint32_t)__shfl_xor(mx, off, 64));
    if (lane == 0) {
      a.q_cost[qi] = fits ? mx : (uint32_t)cnt;
      if (!fits) a.q_flag[qi] = 1u;
    }
    a.lane_range[(size_t)qi * 64 + lane] = fits ? make_uint2((uint32_t)qbase + (incl - tot), tot) : make_uint2(0u, 0u);
  }
  if (!fits) {
    for (int c = wave; c < nch; c += nw) a.frag_off[base + (size_t)c * 64] = kNoFrag;
    return;
  }
  uint32_t run = (uint32_t)qbase + (incl - tot);
  for (int t0 = 0; t0 < nch; t0 += step) {
    const int c0 = t0 + wave * kU;
    if (nch > step) {  // more than one step: the masks again
      load_masks(c0);
      n = 0;
#pragma unroll
      for (int k = 0; k < kU; ++k) {
        mk[k] = c0 + k < cut ? mk[k] : 0ull;
        n += (uint32_t)__popcll(mk[k]);
      }
      sync();  // the last step's counts are read
      s_n[wave][lane] = n;
      sync();
    }
    uint32_t at = run, step_n = n;
    if (nw > 1) {
      step_n = 0;
#pragma unroll
      for (int w = 0; w < kPoWaves; ++w) {
        if (w == wave) at = run + step_n;
        step_n += s_n[w][lane];
      }
    }
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      if (c0 + k < nch) a.frag_off[base + (size_t)(c0 + k) * 64] = at;
      at += (uint32_t)__popcll(mk[k]);
    }
    run += step_n;
  }
}

// Orders the quadrants by decreasing cost (64 logarithmic buckets, one
// 1024-lane workgroup), so the blend kernels dispatch the longest per-pixel
// chains first and the tail of the launch is short work.  The order within a
// bucket is arbitrary; each quadrant's result does not depend on it.
// counters[kCostClass + i] receives the number of quadrants whose cost is at
// least 256, 64, 32, 16 and 1 (i = 0..kSegLog), which come first in the order
// in that order.  host (pinned memory, may be null) receives counters[0..8], final from
// the pair-offset pass on.
__global__ __launch_bounds__(1024) void k_order_quads(int nq, const uint32_t* cost, uint32_t* order,
                                                      uint32_t* counters, uint32_t* host) {
  __shared__ uint32_t s_cnt[64], s_base[64];
  const int tid = threadIdx.x;
  if (host != nullptr && tid < 9) host[tid] = counters[tid];
  if (tid < 64) s_cnt[tid] = 0;
  __syncthreads();
  auto bucket = [](uint32_t c) {  // 63 for the costliest
    const int lg = c == 0u ? 0 : 32 - __clz(c);  // 1 + floor(log2 c)
    int b = lg * 2 + (lg >= 2 ? (int)((c >> (lg - 2)) & 1u) : 0);
    return 63 - min(b, 63);
  };
  // Most quadrants are empty (cost 0, the last bucket): a wave counts and
  // places those with one LDS atomic instead of one per lane.
  const int lane = tid & 63;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  constexpr int kU = 8;  // costs in flight a lane
  auto each = [&](auto&& fn) {  // fn(quadrant or nq and more, its cost), the whole wave at once
    for (int i0 = 0; i0 < nq; i0 += 1024 * kU) {  // uniform
      uint32_t c[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) c[u] = cost[min(i0 + u * 1024 + tid, nq - 1)];
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (i0 + u * 1024 < nq) fn(i0 + u * 1024 + tid, c[u]);
    }
  };
  each([&](int i, uint32_t c) {
    const uint64_t zero = __ballot(i < nq && c == 0u);
    if (lane == 0 && zero) atomicAdd(&s_cnt[63], (uint32_t)__popcll(zero));
    if (i < nq && c != 0u) atomicAdd(&s_cnt[bucket(c)], 1u);
  });
  __syncthreads();
  if (tid < 64) {
    uint32_t incl = s_cnt[tid];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)incl, off);
      if (lane >= off) incl += y;
    }
    s_base[tid] = incl - s_cnt[tid];
    // two buckets an octave: costs of 2^k and more are in 0..61 - 2 k
    const int c = tid == 45 ? 0 : tid == 49 ? 1 : tid == 51 ? 2 : tid == 53 ? 3 : tid == 62 ? 4 : -1;
    if (c >= 0) counters[kCostClass + c] = incl;
  }
  __syncthreads();
  each([&](int i, uint32_t c) {
    const uint64_t zero = __ballot(i < nq && c == 0u);
    uint32_t zbase = 0;
    if (lane == 0 && zero) zbase = atomicAdd(&s_base[63], (uint32_t)__popcll(zero));
    zbase = (uint32_t)__shfl((int)zbase, 0);
    if (i < nq) {
      if (c == 0u) order[zbase + (uint32_t)__popcll(zero & lt)] = (uint32_t)i;
      else order[atomicAdd(&s_base[bucket(c)], 1u)] = (uint32_t)i;
    }
  });
}

hipError_t launch_order_quads(int nq, const uint32_t* cost, uint32_t* order, uint32_t* counters,
                              uint32_t* host, hipStream_t s) {
  if (nq <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_order_quads, dim3(1), dim3(1024), 0, s, nq, cost, order, counters, host);
  return hipGetLastError();
}

__global__ void k_iota_u32(uint32_t* p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = (uint32_t)i;
}

hipError_t launch_iota_u32(uint32_t* p, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_iota_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t launch_pair_offsets(const AcceptArgs& a, hipStream_t s) {
  if (a.vs.T == 0) return hipSuccess;
  hipLaunchKernelGGL(k_pair_offsets, dim3((unsigned)(a.vs.T * quads_per_tile(a.vs.B))), dim3(kPoWaves * 64), 0, s, a);
  return hipGetLastError();
}

// Pair-store fill: balanced like the acceptance pass, one wave per
// (quadrant, chunk).  The chunk's accepted pairs are dealt out 64 per step
// in pixel order (SlotOwner names the pixel of every pair slot; the
// slot's rank among the pixel's pairs picks the entry from the pixel's mask
// bits), so consecutive lanes write consecutive records of a pixel's run.
// Each lane recomputes its pair and stores the entry data the blend chains
// need.  Bound by its 40 bytes a pair: 71 us for 300k surfels at 800 x 600 and
// 257 for 1M at 1237 x 823, with 48 bytes 79 and 290 (232 MB written and 71 read
// at 800 x 600, 3.8 TB/s; a large copy reaches 4.8).
template <bool kPart>
__global__ __launch_bounds__(64) void k_pair_write(AcceptArgs a) {
  __shared__ float4 s_q0[64], s_q1[64], s_q2[64], s_q3[64], s_q4[64];
  __shared__ uint32_t s_pos[64];
  __shared__ unsigned long long s_mask[64];
  __shared__ uint32_t s_start[64], s_foff[64];
  __shared__ uint32_t s_head[64];
  __shared__ uint32_t s_rid[kPart ? 64 : 1];
  const int lane = threadIdx.x;
  if (a.counters[1] & kErrCapacity) return;
  const uint32_t nwork = *a.work_count;
  for (uint32_t w = blockIdx.x; w < nwork; w += gridDim.x) {
    const WorkItem it = unpack_work(a.work[nwork - 1u - w]);  // from the end: see work_capacity
    if (a.q_flag[it.qi] != 0u) continue;
    const int qx0 = it.x0, qy0 = it.y0;
    // lane as pixel: its accepted pairs of the chunk and where they go
    const size_t slot = it.first + 64u * (size_t)it.qi + lane;
    const uint64_t mm = a.masks[slot];
    const uint32_t foff = mm ? a.frag_off[slot] : 0u;
    const uint32_t n = (uint32_t)__popcll(mm);
    uint32_t incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t v = (uint32_t)__shfl_up((int)incl, off, 64);
      if (lane >= off) incl += v;
    }
    const uint32_t total = (uint32_t)__shfl((int)incl, 63, 64);
    if (total == 0u) continue;  // uniform across the wave
    wave_lds_fence();  // the previous item's readers are done
    const uint32_t first = incl - n;
    s_mask[lane] = mm;
    s_start[lane] = first;
    s_foff[lane] = foff;
    if ((uint32_t)lane < it.m) {
      const uint2 v = a.sub[it.first + lane];
      const float4* rc = a.rec + (size_t)kRecQuads * v.x;
      s_q0[lane] = rc[0];
      s_q1[lane] = rc[1];
      s_q2[lane] = rc[2];
      s_q3[lane] = rc[3];
      s_q4[lane] = rc[4];
      s_pos[lane] = v.y;
      if (kPart) s_rid[lane] = v.x;
    }
    wave_lds_fence();
    SlotOwner owner;
    for (uint32_t base = 0; base < total; base += 64) {
      const uint32_t t = base + (uint32_t)lane;
      const int p = (int)owner.at(s_head, base, first, n);
      if (t >= total) continue;
      const uint32_t k = t - s_start[p];
      const int j = select_bit(s_mask[p], k);
      Pair e;
      eval_pair<false>(pixel_centre<kPart>(qx0 + (p & 7)), pixel_centre<kPart>(qy0 + (p >> 3)), s_q0[j], s_q1[j],
                       s_q2[j], 0.0f, e);
      const float4 q3 = s_q3[j], q4 = s_q4[j];
      // the distortion weight m(depth), as the blends form it
      const float m_d = dist_weight<kPart>(e.depth);
      char* pr = a.ps.rec + (size_t)PairLayout<kPart>::kBytes * (size_t)(s_foff[p] + k);
      float4* q = reinterpret_cast<float4*>(pr);
      q[0] = make_float4(m_d, __uint_as_float(kPart ? s_rid[j] : s_pos[j]), e.alpha, e.depth);
      q[1] = make_float4(q3.w, q4.x, q4.y, q3.x);
      if (kPart) q[2] = make_float4(q3.y, q3.z, __uint_as_float(s_pos[j]), 0.0f);
      else *reinterpret_cast<float2*>(pr + 32) = make_float2(q3.y, q3.z);
    }
  }
}

hipError_t launch_pair_write(const AcceptArgs& a, size_t max_items, hipStream_t s) {
  if (max_items == 0) return hipSuccess;
  const unsigned grid = (unsigned)(max_items < kChunkBlocks ? max_items : kChunkBlocks);
  if (a.part) hipLaunchKernelGGL(k_pair_write<true>, dim3(grid), dim3(64), 0, s, a);
  else hipLaunchKernelGGL(k_pair_write<false>, dim3(grid), dim3(64), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Forward blend, dsr/cuda_rasterizer/forward.cu:256-441.  One wave64 per
// 8 x 8 quadrant; each lane walks, front to back, only the entries its
// acceptance mask marks, recomputing each pair exactly and applying the
// reference's update.  Entries a lane skips are the ones the reference
// skips, so T, the accumulators and the contributor counts (positions in the
// full tile list) come out bit-identical.
// ---------------------------------------------------------------------------
#ifndef SR_FWD_PREFETCH
#define SR_FWD_PREFETCH 8
#endif
constexpr int kPre = SR_FWD_PREFETCH;  // stored pairs of a pixel per batch
constexpr int kPreGroup = 4;           // loaded or not together
static_assert(kPre % kPreGroup == 0 && kPre <= kPairPad, "whole groups, reads past the last pair within the padding");
using V3 = float __attribute__((ext_vector_type(3)));
template <class T> SR_DEV T load4(const char* p) {  // from a 4-byte aligned place
  T v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, 4), sizeof(float) * (sizeof(T) == 16 ? 3 : sizeof(T) / 4));
  return v;
}

// Forward blend of a quadrant whose pairs missed the store: the records staged
// chunk by chunk, the pairs recomputed, lane = pixel.
template <bool kPart>
SR_DEV void blend_fwd_missed(const BlendArgs& a, int qi) {
  __shared__ float4 s_q0[64], s_q1[64], s_q2[64], s_q3[64], s_q4[64];
  __shared__ uint32_t s_pos[64];
  __shared__ uint32_t s_rid[kPart ? 64 : 1];
  const int B = a.vs.B, QX = B / kQuad, Q = QX * QX;
  const int tile = qi / Q, q = qi % Q;
  const ViewInfo& vi = a.vs.v[view_of_tile(a.vs, (uint32_t)tile)];
  const int lt = tile - (int)vi.tile_base;
  const int tx = lt % vi.gx, ty = lt / vi.gx;
  const int lane = threadIdx.x;
  const int pix = lane;  // of the quadrant
  const uint32_t pxi = (uint32_t)(tx * B + (q % QX) * kQuad + (pix & 7));
  const uint32_t pyi = (uint32_t)(ty * B + (q / QX) * kQuad + (pix >> 3));
  const bool inside = pxi < (uint32_t)vi.W && pyi < (uint32_t)vi.H;
  bool done = !inside;
  const uint32_t rbeg = a.ranges[2 * tile], ntile = a.ranges[2 * tile + 1] - rbeg;
  const int cnt = (int)a.sub_count[qi];
  const uint2* list = a.sub + (size_t)Q * rbeg + (size_t)q * ntile;
  const uint64_t* masks = a.masks + mask_base(Q, rbeg, ntile, tile, q);
  const uint32_t* frag_off = a.frag_off + mask_base(Q, rbeg, ntile, tile, q);
  const float pixx = pixel_centre<kPart>((int)pxi), pixy = pixel_centre<kPart>((int)pyi);
  float T = 1.0f;
  uint32_t last_contributor = 0;
  float Sem[kPart ? kMaxSem : 1];
#pragma unroll
  for (int ch = 0; ch < (kPart ? kMaxSem : 1); ++ch) Sem[ch] = 0.0f;
  float median_weight = 0.0f;
  float C0 = 0.0f, C1 = 0.0f, C2 = 0.0f, N0 = 0.0f, N1 = 0.0f, N2 = 0.0f;
  float D = 0.0f, M1 = 0.0f, M2 = 0.0f, distortion = 0.0f, median_depth = 0.0f, median_contributor = -1.0f;
  int blended = 0;
  const int nch = (cnt + 63) / 64;
  // One front-to-back step of the reference's update (forward.cu:383-415);
  // false once T would drop below 1e-4 (the pixel is done).  mm is the
  // distortion weight mcoef (1 - near / depth).
  auto step = [&](float alpha, float depth, float mm, uint32_t pos, const float4& nc, float g, float bl,
                  uint32_t rid) -> bool {
    const float test_T = T * (1.0f - alpha);
    if (test_T < 0.0001f) return false;
    const uint32_t contributor = pos + 1u;
    const float w = alpha * T;
    const float A = 1.0f - T;
    auto weighed = [&](float x) { return kPart ? (x * alpha) * T : x * w; };
    distortion += weighed(((mm * mm) * A + M2) - (2.0f * mm) * M1);
    D += weighed(depth);
    M1 += weighed(mm);
    M2 += weighed(mm * mm);
    if (T > 0.5f) {
      median_depth = depth;
      median_weight = w;
      median_contributor = (float)contributor;
    }
    N0 += weighed(nc.x);
    N1 += weighed(nc.y);
    N2 += weighed(nc.z);
    C0 += weighed(nc.w);
    C1 += weighed(g);
    C2 += weighed(bl);
    if (kPart) {
      const float* sr = a.sem + (size_t)rid * a.S;
#pragma unroll
      for (int ch = 0; ch < kMaxSem; ++ch)
        if (ch < a.S) Sem[ch] += weighed(sr[ch]);
    }
    T = test_T;
    last_contributor = contributor;
    ++blended;
    return true;
  };
  {
    // Some chunk missed the store: stage the records chunk by chunk and
    // recompute the pairs of chunks without stored pairs.
    ChunkRegs nx{};
    uint2 v2 = make_uint2(0u, 0u);
    if (nch > 0) {
      nx = chunk_load(masks, frag_off, a.rec, lane, 0, chunk_entry(list, cnt, lane, 0, nch));
      v2 = chunk_entry(list, cnt, lane, 1, nch);
    }
    for (int c = 0; c < nch; ++c) {
      const int m = min(64, cnt - c * 64);
      uint64_t mask = done ? 0ull : nx.mask;
      __syncthreads();
      if (lane < m) {
        s_pos[lane] = nx.v.y;
        if (kPart) s_rid[lane] = nx.v.x;
        s_q0[lane] = nx.q0;
        s_q1[lane] = nx.q1;
        s_q2[lane] = nx.q2;
        s_q3[lane] = nx.q3;
        s_q4[lane] = nx.q4;
      }
      __syncthreads();
      if (c + 1 < nch) {  // in flight while this chunk blends
        const uint2 ve = v2;
        v2 = chunk_entry(list, cnt, lane, c + 2, nch);
        nx = chunk_load(masks, frag_off, a.rec, lane, c + 1, ve);
      }
      if (__ballot(mask != 0ull) == 0ull) continue;
      while (mask != 0ull) {
        const int j = __builtin_ctzll(mask);
        mask &= mask - 1ull;
        float alpha, depth;
        Pair e;  // none of the quadrant's pairs is stored
        if (!eval_pair<false>(pixx, pixy, s_q0[j], s_q1[j], s_q2[j], 0.0f, e)) continue;
        alpha = e.alpha;
        depth = e.depth;
        const float4 q3 = s_q3[j], q4 = s_q4[j];
        if (!step(alpha, depth, dist_weight<kPart>(depth), s_pos[j], q3, q4.x, q4.y, kPart ? s_rid[j] : 0u)) {
          done = true;
          break;
        }
      }
      if (__ballot(!done) == 0ull) break;
    }
  }
  if (inside) {
    const size_t HW = (size_t)vi.H * vi.W, pid = (size_t)vi.W * pyi + pxi, pb = vi.pix_base;
    float* final_T = a.final_T + 3 * pb;
    uint32_t* n_contrib = a.n_contrib + 2 * pb;
    float* out_color = a.out_color + 3 * pb;
    float* out_others = a.out_others + (kPart ? 8 : 7) * pb;
    if (kPart) {
      out_others[pid + 7 * HW] = median_weight;
      float* out_sem = a.out_sem + (size_t)a.S * pb;
#pragma unroll
      for (int ch = 0; ch < kMaxSem; ++ch)
        if (ch < a.S) out_sem[ch * HW + pid] = Sem[ch];
    }
    final_T[pid] = T;
    n_contrib[pid] = last_contributor;
    out_color[pid] = C0 + T * a.bg[0];
    out_color[HW + pid] = C1 + T * a.bg[1];
    out_color[2 * HW + pid] = C2 + T * a.bg[2];
    n_contrib[pid + HW] = f2u(median_contributor);
    final_T[pid + HW] = M1;
    final_T[pid + 2 * HW] = M2;
    out_others[pid] = D;
    out_others[pid + HW] = 1.0f - T;
    out_others[pid + 2 * HW] = N0;
    out_others[pid + 3 * HW] = N1;
    out_others[pid + 4 * HW] = N2;
    out_others[pid + 5 * HW] = median_depth;
    out_others[pid + 6 * HW] = distortion;
    // the backward cuts the pixel's run into the same segments as a stored run
    a.lane_range[(size_t)qi * 64 + pix].y = (uint32_t)blended;
  }
}

// Forward blend of the quadrants whose pairs are all in the store, each
// pixel's pairs one contiguous run in entry order.  A wave takes 16 pixels
// with 4 lanes each; the 4 lanes of a pixel walk the same run in step (each
// runs the transmittance update, so all agree on where the pixel stops) and
// split the accumulators: role 0 M1, M2 and distortion, role 1 the normal, role
// 2 the colour, role 3 the depth.  Every lane executes the same
// instructions (role values are picked by select), so the serial chain of a
// long pixel costs a quarter of the full update per pair; each accumulator
// sees exactly the reference's operations in order.
// What bounds it is that chain: a run of hundreds of pairs is blended at the
// rate one wave issues.  So a batch first runs the transmittances alone (two
// operations a pair; they only fall, so the last one tells whether the pixel
// saturates in the batch), and where every pixel of the wave has a whole
// batch left and none saturates, the updates go in without per-pair
// conditions.  The last contributor and the median are pairs of the run, looked
// up once at its end from their counts.  300k surfels: 61 us at 800 x 600 and
// 78 at 400 x 300, where conditions on every pair and 20 pairs a batch, copied
// from the prefetch registers (185 a lane, two waves a SIMD), took 94 and 122.
// Batches of 12 and 16 pairs: 63, 69 and 84, 81 us.
// The _part variant sums its outputs as (value * alpha) * T (its kernel's
// expression; the plain one adds value * (alpha * T)), keeps the median pair's
// weight and leaves each pair's T in fW, which the backward overwrites only
// later, for the semantic pass.
template <bool kPart>
__global__ __launch_bounds__(64) void k_blend_fwd(BlendArgs a) {
  static_assert(kSplit == 4, "4 waves of 16 pixels x 4 roles per quadrant");
  if (a.counters[1] & kErrCapacity) return;
  const int qi = (int)a.q_order[blockIdx.x / kSplit], part = blockIdx.x % kSplit;
  if (a.q_flag[qi] != 0u) {
    if (part == 0) blend_fwd_missed<kPart>(a, qi);
    return;
  }
  const int B = a.vs.B, QX = B / kQuad, Q = QX * QX;
  const int tile = qi / Q, q = qi % Q;
  const ViewInfo& vi = a.vs.v[view_of_tile(a.vs, (uint32_t)tile)];
  const int lt = tile - (int)vi.tile_base;
  const int tx = lt % vi.gx, ty = lt / vi.gx;
  const int lane = threadIdx.x, role = lane & 3;
  const int pix = part * 16 + (lane >> 2);
  const uint32_t pxi = (uint32_t)(tx * B + (q % QX) * kQuad + (pix & 7));
  const uint32_t pyi = (uint32_t)(ty * B + (q / QX) * kQuad + (pix >> 3));
  const bool inside = pxi < (uint32_t)vi.W && pyi < (uint32_t)vi.H;
  const int cnt = (int)a.sub_count[qi];
  // lane_range is written by the pair-offset pass, which runs only when the
  // view has instances: read it for non-empty quadrants only
  const uint2 rg = (inside && cnt > 0) ? a.lane_range[(size_t)qi * 64 + pix] : make_uint2(0u, 0u);
  // Each lane loads three words of a record: role 0 (m, .., alpha), role 1 the
  // normal, role 2 the colour and role 3 (depth, .., ..); alpha reaches the
  // other lanes of the pixel from role 0 by a quad broadcast.  A lane sums its
  // words in a0..a2, except that role 0 has m^2 for the second, and the
  // distortion in a2.
  constexpr int kBytes = PairLayout<kPart>::kBytes;
  const char* run = a.ps.rec + (size_t)kBytes * rg.x + (role == 0 ? 0 : role == 1 ? 28 : role == 2 ? 16 : 12);
  float T = 1.0f;
  float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, median_weight = 0.0f;
  float* pair_T = kPart && a.S > 0 ? reinterpret_cast<float*>(a.ps.fW) + rg.x : nullptr;
  int blended = 0, in_front = 0;  // pairs blended; those with T above 1/2
  bool done = false;
  int left = (int)rg.y;
  // whole groups, so up to kPreGroup - 1 pairs past the run (nothing uses
  // them; the store is padded)
  auto fetch = [&](V3 (&b)[kPre], const char* at, int n) {
#pragma unroll
    for (int g = 0; g < kPre; g += kPreGroup)
      if (g < n) {
#pragma unroll
        for (int k = g; k < g + kPreGroup; ++k) b[k] = load4<V3>(at + kBytes * k);
      }
  };
  // forward.cu:383-415 for one pair
  auto update = [&](const V3& v, float alpha, float Tk) {
    const float w = alpha * Tk;
    const float A = 1.0f - Tk;
    // role 0: the distortion term (m^2 A + M2 - 2 m M1), a0 = M1, a1 = M2
    const float x1 = role == 0 ? v.x * v.x : v.y;
    const float x2 = role == 0 ? (x1 * A + a1) - (2.0f * v.x) * a0 : v.z;
    auto weighed = [&](float x) { return kPart ? (x * alpha) * Tk : x * w; };
    a0 += weighed(v.x);
    a1 += weighed(x1);
    a2 += weighed(x2);
    if (kPart && Tk > 0.5f) median_weight = w;
  };
  auto blend = [&](const V3 (&b)[kPre]) {
    const int n = min(left, kPre);
    float Tk[kPre + 1];
    Tk[0] = T;
#pragma unroll
    for (int k = 0; k < kPre; ++k) Tk[k + 1] = Tk[k] * (1.0f - quad_bcast0(b[k].z));
    if (kPart && pair_T != nullptr) {
      // a quarter of the batch a lane; behind a saturating pair nobody reads it
#pragma unroll
      for (int u = 0; u < kPre / 4; ++u) {
        const float x = role < 2 ? (role == 0 ? Tk[u] : Tk[kPre / 4 + u])
                                 : (role == 2 ? Tk[kPre / 2 + u] : Tk[3 * kPre / 4 + u]);
        const int k = role * (kPre / 4) + u;
        if (k < n) pair_T[blended + k] = x;
      }
    }
    if (__ballot(n < kPre || !(Tk[kPre] >= 0.0001f)) == 0ull) {  // of the lanes with pairs left
#pragma unroll
      for (int k = 0; k < kPre; ++k) {
        update(b[k], quad_bcast0(b[k].z), Tk[k]);
      }
      if (__ballot(T > 0.5f) != 0ull) {
#pragma unroll
        for (int k = 0; k < kPre; ++k) in_front += Tk[k] > 0.5f ? 1 : 0;
      }
      blended += kPre;
      T = Tk[kPre];
    } else {
#pragma unroll
      for (int k = 0; k < kPre; ++k) {
        if (k < n && !done) {
          if (Tk[k + 1] < 0.0001f) {
            done = true;
          } else {
            update(b[k], quad_bcast0(b[k].z), Tk[k]);
            in_front += Tk[k] > 0.5f ? 1 : 0;
            T = Tk[k + 1];
            ++blended;
          }
        }
      }
    }
    left -= kPre;
  };
  V3 b0[kPre] = {}, b1[kPre] = {};
  fetch(b0, run, left);
  while (left > 0 && !done) {  // the four lanes of a pixel share left and done
    run += kBytes * kPre;
    fetch(b1, run, left - kPre);  // in flight while b0 blends
    blend(b0);
    if (left > 0 && !done) {
      run += kBytes * kPre;
      fetch(b0, run, left - kPre);
      blend(b1);
    }
  }
  if (!inside) return;
  const size_t HW = (size_t)vi.H * vi.W, pid = (size_t)vi.W * pyi + pxi, pb = vi.pix_base;
  float* final_T = a.final_T + 3 * pb;
  float* out_color = a.out_color + 3 * pb;
  float* out_others = a.out_others + (kPart ? 8 : 7) * pb;
  if (role == 0) {
    final_T[pid + HW] = a0;
    final_T[pid + 2 * HW] = a1;
    out_others[pid + 6 * HW] = a2;  // the distortion
    if (kPart) out_others[pid + 7 * HW] = median_weight;
  } else if (role == 1) {
    out_others[pid + 2 * HW] = a0;
    out_others[pid + 3 * HW] = a1;
    out_others[pid + 4 * HW] = a2;
  } else if (role == 2) {
    out_color[pid] = a0 + T * a.bg[0];
    out_color[HW + pid] = a1 + T * a.bg[1];
    out_color[2 * HW + pid] = a2 + T * a.bg[2];
  } else {
    out_others[pid] = a0;  // the depth
    const char* first = a.ps.rec + (size_t)kBytes * rg.x;
    auto word = [&](int n, int byte) { return *reinterpret_cast<const uint32_t*>(first + (size_t)kBytes * (n - 1) + byte); };
    auto contributor = [&](int n) { return word(n, kPart ? 40 : 4) + 1u; };  // tile position
    uint32_t* n_contrib = a.n_contrib + 2 * pb;
    final_T[pid] = T;
    n_contrib[pid] = blended > 0 ? contributor(blended) : 0u;
    n_contrib[pid + HW] = f2u(in_front > 0 ? (float)contributor(in_front) : -1.0f);
    out_others[pid + HW] = 1.0f - T;
    out_others[pid + 5 * HW] = in_front > 0 ? __uint_as_float(word(in_front, 12)) : 0.0f;
    // the backward passes walk only the blended prefix of the run
    if (cnt > 0) a.lane_range[(size_t)qi * 64 + pix].y = (uint32_t)blended;
  }
}

hipError_t launch_blend_fwd(const BlendArgs& a, hipStream_t s) {
  if (a.vs.T == 0) return hipSuccess;
  if (a.vs.B != 8 && a.vs.B != 16 && a.vs.B != 32) return hipErrorInvalidValue;
  const unsigned nblk = (unsigned)(a.vs.T * quads_per_tile(a.vs.B));
  if (a.part) hipLaunchKernelGGL(k_blend_fwd<true>, dim3(nblk * kSplit), dim3(64), 0, s, a);
  else hipLaunchKernelGGL(k_blend_fwd<false>, dim3(nblk * kSplit), dim3(64), 0, s, a);
  return hipGetLastError();
}

// Semantic channels of the _part variant (dsp/cuda_rasterizer/forward.cu:417):
// Sem[ch] += (s[ch] alpha) T over the pixel's blended pairs in order, with
// the T the blend left per pair.  kLanes lanes per pixel, one channel each:
// a pair's alpha and T are one broadcast load and its semantics one row
// gather, and only the sum itself is serial, so kSemPre pairs' loads are in
// flight.  One wave per 64 / kLanes pixels, quadrants longest chain first.
// Memory-bound: 20 + 4 S bytes a pair.
constexpr int kSemPre = 8;
template <int kLanes>
__global__ __launch_bounds__(64) void k_blend_semantics(BlendArgs a) {
  constexpr int kWaves = kLanes, kPix = 64 / kLanes;  // waves per quadrant, pixels per wave
  const int B = a.vs.B, QX = B / kQuad, Q = QX * QX;
  if (a.counters[1] & kErrCapacity) return;
  const int qi = (int)a.q_order[blockIdx.x / kWaves], wv = blockIdx.x % kWaves;
  if (a.q_flag[qi] != 0u) return;  // blended with the quadrant's recomputed pairs
  const int tile = qi / Q, q = qi % Q;
  const ViewInfo& vi = a.vs.v[view_of_tile(a.vs, (uint32_t)tile)];
  const int lt = tile - (int)vi.tile_base;
  const int lane = threadIdx.x, ch = lane % kLanes, pix = wv * kPix + lane / kLanes;
  const uint32_t pxi = (uint32_t)((lt % vi.gx) * B + (q % QX) * kQuad + (pix & 7));
  const uint32_t pyi = (uint32_t)((lt / vi.gx) * B + (q / QX) * kQuad + (pix >> 3));
  if (pxi >= (uint32_t)vi.W || pyi >= (uint32_t)vi.H || ch >= a.S) return;
  float sum = 0.0f;
  if (a.sub_count[qi] > 0u) {
    const uint2 rg = a.lane_range[(size_t)qi * 64 + pix];
    const float* pair_T = reinterpret_cast<const float*>(a.ps.fW);
    for (uint32_t i = 0; i < rg.y; i += kSemPre) {
      V3 p0[kSemPre];  // m, surfel, alpha
      float T[kSemPre], sv[kSemPre];
#pragma unroll
      for (int k = 0; k < kSemPre; ++k) {  // past the run's end: its last pair again, not summed
        const size_t f = rg.x + min(i + (uint32_t)k, rg.y - 1u);
        p0[k] = load4<V3>(a.ps.rec + (size_t)PairLayout<true>::kBytes * f);
        T[k] = pair_T[f];
      }
#pragma unroll
      for (int k = 0; k < kSemPre; ++k) sv[k] = a.sem[(size_t)__float_as_uint(p0[k].y) * a.S + ch];
#pragma unroll
      for (int k = 0; k < kSemPre; ++k)
        if (i + (uint32_t)k < rg.y) sum += (sv[k] * p0[k].z) * T[k];
    }
  }
  const size_t HW = (size_t)vi.H * vi.W;
  a.out_sem[(size_t)a.S * vi.pix_base + ch * HW + (size_t)vi.W * pyi + pxi] = sum;
}

hipError_t launch_blend_semantics(const BlendArgs& a, hipStream_t s) {
  if (a.vs.T == 0 || a.S <= 0) return hipSuccess;
  const unsigned nq = (unsigned)(a.vs.T * quads_per_tile(a.vs.B));
  if (a.S <= 4) hipLaunchKernelGGL(k_blend_semantics<4>, dim3(nq * 4), dim3(64), 0, s, a);
  else if (a.S <= 8) hipLaunchKernelGGL(k_blend_semantics<8>, dim3(nq * 8), dim3(64), 0, s, a);
  else hipLaunchKernelGGL(k_blend_semantics<16>, dim3(nq * 16), dim3(64), 0, s, a);
  return hipGetLastError();
}

// markVisible / checkFrustum, rasterizer_impl.cu:54-66.
__global__ void k_mark_visible(int P, const float* means3D, const float* vm, uint8_t* present) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P) return;
  const float m0 = means3D[3 * i], m1 = means3D[3 * i + 1], m2 = means3D[3 * i + 2];
  const float vz = ((vm[2] * m0 + vm[6] * m1) + vm[10] * m2) + vm[14];
  present[i] = vz <= 0.2f ? 0 : 1;
}

hipError_t launch_mark_visible(int P, const float* means3D, const float* vm, uint8_t* present,
                               hipStream_t s) {
  if (P == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mark_visible, dim3((P + 255) / 256), dim3(256), 0, s, P, means3D, vm, present);
  return hipGetLastError();
}

// Copies the instance count and the error flags to a caller-visible status
// word, so batched callers can check capacity without reading internal state.
__global__ void k_copy_status(const uint32_t* counters, uint32_t* status) {
  if (threadIdx.x < 9) status[threadIdx.x] = counters[threadIdx.x];
}

hipError_t launch_copy_status(const uint32_t* counters, uint32_t* status, hipStream_t s) {
  hipLaunchKernelGGL(k_copy_status, dim3(1), dim3(64), 0, s, counters, status);
  return hipGetLastError();
}

}  // namespace sr
