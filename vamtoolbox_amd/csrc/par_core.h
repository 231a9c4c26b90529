// Device-level cores of the parallel-beam operators, shared by the plain
// kernels (parallel.hip), the fused BCLP kernels (bclp.hip) and the batched
// launch (batched.hip).
//
// Discretisation: the reference's CPU projector "D1"
// (vamtoolbox/projector/Projector3DParallel.py:113-207) plus the detector
// offset / absorption / inclination extensions.  Layouts: volume (n, n, nz)
// and sinogram (n, n_angles, nz), both z-contiguous; a lane owns one ray or
// voxel column and ZV consecutive z values, so sample weights are identical
// across a wavefront and every tap is a coalesced load.
//
// Geometry (sample coordinates, floor/ceil decisions, weights) is evaluated
// in float64 with the reference's operation order (translation units are
// compiled with -ffp-contract=off) so that every discontinuous decision
// matches the reference; data arithmetic is float32 with explicit fused
// multiply-adds.  No core uses atomics.
#pragma once

#include <type_traits>

#include "vamx_internal.h"

namespace vamx {

template <int ZV> struct VecT;
template <> struct VecT<1> { using T = float; };
template <> struct VecT<2> { using T = float2; };
template <> struct VecT<3> { using T = float3; };
template <> struct VecT<4> { using T = float4; };

template <int ZV> __device__ __forceinline__ typename VecT<ZV>::T vzero();
template <> __device__ __forceinline__ float vzero<1>() { return 0.0f; }
template <> __device__ __forceinline__ float2 vzero<2>() { return make_float2(0.f, 0.f); }
template <> __device__ __forceinline__ float3 vzero<3>() { return make_float3(0.f, 0.f, 0.f); }
template <> __device__ __forceinline__ float4 vzero<4>() { return make_float4(0.f, 0.f, 0.f, 0.f); }

template <int ZV> __device__ __forceinline__ typename VecT<ZV>::T vload(const float* p);
template <> __device__ __forceinline__ float vload<1>(const float* p) { return *p; }
template <> __device__ __forceinline__ float2 vload<2>(const float* p) { return *reinterpret_cast<const float2*>(p); }
template <> __device__ __forceinline__ float4 vload<4>(const float* p) { return *reinterpret_cast<const float4*>(p); }

// Buffer loads: a wave-uniform base in a buffer descriptor (scalar
// registers) plus a per-lane byte offset and a scalar byte offset, so the
// per-load address arithmetic is scalar work.  The descriptor covers
// `bytes` from the base (raw buffer, no stride); word 3 is the gfx9 raw
// 32-bit data format.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const float* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
}
template <int ZV>
__device__ __forceinline__ typename VecT<ZV>::T bload(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff);
template <>
__device__ __forceinline__ float bload<1>(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
}
template <>
__device__ __forceinline__ float2 bload<2>(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0);
  return make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
}
template <>
__device__ __forceinline__ float4 bload<4>(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0);
  return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}

template <int ZV> __device__ __forceinline__ void vstore(float* p, typename VecT<ZV>::T v);
template <> __device__ __forceinline__ void vstore<1>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void vstore<2>(float* p, float2 v) { *reinterpret_cast<float2*>(p) = v; }
template <> __device__ __forceinline__ void vstore<4>(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }

__device__ __forceinline__ float vfma(float a, float x, float y) { return __builtin_fmaf(a, x, y); }
__device__ __forceinline__ float4 vfma(float a, float4 x, float4 y) {
  return make_float4(__builtin_fmaf(a, x.x, y.x), __builtin_fmaf(a, x.y, y.y), __builtin_fmaf(a, x.z, y.z),
                     __builtin_fmaf(a, x.w, y.w));
}
__device__ __forceinline__ float2 vfma(float a, float2 x, float2 y) {
  return make_float2(__builtin_fmaf(a, x.x, y.x), __builtin_fmaf(a, x.y, y.y));
}
__device__ __forceinline__ float3 vfma(float a, float3 x, float3 y) {
  return make_float3(__builtin_fmaf(a, x.x, y.x), __builtin_fmaf(a, x.y, y.y), __builtin_fmaf(a, x.z, y.z));
}
__device__ __forceinline__ float3 vmul(float a, float3 x) { return make_float3(a * x.x, a * x.y, a * x.z); }
__device__ __forceinline__ float vmul(float a, float x) { return a * x; }
__device__ __forceinline__ float2 vmul(float a, float2 x) { return make_float2(a * x.x, a * x.y); }
__device__ __forceinline__ float4 vmul(float a, float4 x) { return make_float4(a * x.x, a * x.y, a * x.z, a * x.w); }
__device__ __forceinline__ float vsub(float a, float b) { return a - b; }
__device__ __forceinline__ float4 vsub(float4 a, float4 b) {
  return make_float4(a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w);
}
__device__ __forceinline__ float2 vsub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float vadd(float a, float b) { return a + b; }
__device__ __forceinline__ float2 vadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float3 vadd(float3 a, float3 b) { return make_float3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ float4 vadd(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float clampf(float v, float lo, float hi) { return fminf(fmaxf(v, lo), hi); }
__device__ __forceinline__ float vclamp(float v, float lo, float hi) { return clampf(v, lo, hi); }
__device__ __forceinline__ float2 vclamp(float2 v, float2 lo, float2 hi) {
  return make_float2(clampf(v.x, lo.x, hi.x), clampf(v.y, lo.y, hi.y));
}
__device__ __forceinline__ float4 vclamp(float4 v, float4 lo, float4 hi) {
  return make_float4(clampf(v.x, lo.x, hi.x), clampf(v.y, lo.y, hi.y), clampf(v.z, lo.z, hi.z),
                     clampf(v.w, lo.w, hi.w));
}
__device__ __forceinline__ float3 vclamp(float3 v, float3 lo, float3 hi) {
  return make_float3(clampf(v.x, lo.x, hi.x), clampf(v.y, lo.y, hi.y), clampf(v.z, lo.z, hi.z));
}
__device__ __forceinline__ float vget(float3 v, int q) { return q == 0 ? v.x : (q == 1 ? v.y : v.z); }
__device__ __forceinline__ void vset(float3& v, int q, float x) {
  if (q == 0) v.x = x;
  else if (q == 1) v.y = x;
  else v.z = x;
}
__device__ __forceinline__ float vget(float v, int) { return v; }
__device__ __forceinline__ float vget(float2 v, int q) { return q == 0 ? v.x : v.y; }
__device__ __forceinline__ float vget(float4 v, int q) { return q == 0 ? v.x : (q == 1 ? v.y : (q == 2 ? v.z : v.w)); }
__device__ __forceinline__ void vset(float& v, int, float x) { v = x; }
__device__ __forceinline__ void vset(float2& v, int q, float x) {
  if (q == 0) v.x = x; else v.y = x;
}
__device__ __forceinline__ void vset(float4& v, int q, float x) {
  if (q == 0) v.x = x; else if (q == 1) v.y = x; else if (q == 2) v.z = x; else v.w = x;
}

// absorption weight of a sample at lateral coordinate t and along-ray s:
// exp(-mu * max(0, sqrt(R^2 - t^2) - s) / cos(phi)) inside |t| < R, else 0
// (per-ray form of astra3Dabsorption.getExpabs, astra3Dabsorption.py:129-145)
__host__ __device__ __forceinline__ float abs_weight(const ParDev& g, double t, double s) {
  if (g.mu == 0.0) return 1.0f;
  if (!(fabs(t) < g.radius)) return 0.0f;
  const double half = sqrt(g.radius * g.radius - t * t);
  const double path = fmax(0.0, half - s) * g.inv_cos;
  return expf((float)(-g.mu * path));
}

// np.interp(t, xp, fp, left=0, right=0) with xp[k] = (k - c) - det_offset:
// value = fp[j] + w (fp[j1] - fp[j]); numpy compares t with the end nodes and
// returns fp[-1] exactly at the last node.
__host__ __device__ __forceinline__ bool interp_node(const ParDev& g, double t, int& j, int& j1, float& w) {
  if (!(t >= g.xp0 && t <= g.xp_last)) return false;
  const double u = t - g.xp0;
  int jj = (int)floor(u);
  jj = jj < 0 ? 0 : (jj > g.n - 1 ? g.n - 1 : jj);
  j = jj;
  j1 = jj + 1 < g.n ? jj + 1 : g.n - 1;
  w = (jj == g.n - 1) ? 0.0f : (float)(t - ((double)(jj - g.c) - g.det_offset));
  return true;
}

// weight that a sample at `coord` gives to integer position idx
// (skimage bilinear: floor tap 1-d, ceil tap d; floor == ceil -> 1 + 0)
__device__ __forceinline__ float tap_weight_axis(double coord, int idx) {
  const double f = floor(coord), cl = ceil(coord);
  const double d = coord - f;
  double w = 0.0;
  if ((int)f == idx) w += 1.0 - d;
  if ((int)cl == idx) w += d;
  return (float)w;
}

// ---------------------------------------------------------------------------
// forward projection of ray (k, i) at z .. z+ZV-1, zero inclination
// (Projector3DParallel.py:129-156: warp with matrix R, clip, column sum)
// ---------------------------------------------------------------------------
template <int ZV, bool CLIP>
__device__ __forceinline__ typename VecT<ZV>::T fp_ray(const ParDev& g, const float* __restrict__ vol,
                                                        const float* __restrict__ minmax, int k, int i, int z) {
  using V = typename VecT<ZV>::T;
  const int n = g.n;
  const double* M = g.mats + 6 * i;
  const double M01 = M[1], M02 = M[2], M11 = M[4], M12 = M[5];
  const double kp = (double)k - g.det_offset;
  const double a0 = M[0] * kp, a1 = M[3] * kp;
  const double t = (double)(k - g.c) - g.det_offset;
  V lo = vzero<ZV>(), hi = vzero<ZV>();
  if constexpr (CLIP) {
    lo = vload<ZV>(minmax + z);
    hi = vload<ZV>(minmax + g.nz + z);
  }
  V acc = vzero<ZV>();
  const size_t zstride = (size_t)g.nz;
  // occlusion: slice z+q drops the samples with y = r - c > lim[q]
  // (Projector3DParallel.py:147-153); lim = +inf where no shadow applies
  float lim[ZV];
#pragma unroll
  for (int q = 0; q < ZV; ++q) {
    lim[q] = INFINITY;
    if (g.occ && g.occ_active[(size_t)i * g.nz + z + q]) {
      const float o = g.occ[((size_t)k * g.na + i) * zstride + z + q];
      if (!isnan(o)) lim[q] = o;
    }
  }
  for (int r = 0; r < n; ++r) {
    const double rr = (double)r;
    const double col = (a0 + M01 * rr) + M02;
    const double row = (a1 + M11 * rr) + M12;
    if (!(row > -1.0 && row < (double)n && col > -1.0 && col < (double)n)) continue;
    const double fr = floor(row), fc = floor(col);
    const double dr = row - fr, dc = col - fc;
    const int r0 = (int)fr, c0 = (int)fc;
    const int r1 = (int)ceil(row), c1 = (int)ceil(col);
    const bool vr0 = r0 >= 0, vr1 = r1 < n, vc0 = c0 >= 0, vc1 = c1 < n;
    const float f1dc = (float)(1.0 - dc), fdc = (float)dc;
    const float f1dr = (float)(1.0 - dr), fdr = (float)dr;
    V tl = vzero<ZV>(), tr = vzero<ZV>(), bl = vzero<ZV>(), br = vzero<ZV>();
    if (vr0 && vc0) tl = vload<ZV>(vol + ((size_t)r0 * n + c0) * zstride + z);
    if (vr0 && vc1) tr = vload<ZV>(vol + ((size_t)r0 * n + c1) * zstride + z);
    if (vr1 && vc0) bl = vload<ZV>(vol + ((size_t)r1 * n + c0) * zstride + z);
    if (vr1 && vc1) br = vload<ZV>(vol + ((size_t)r1 * n + c1) * zstride + z);
    const V top = vfma(fdc, tr, vmul(f1dc, tl));
    const V bottom = vfma(fdc, br, vmul(f1dc, bl));
    V v = vfma(fdr, bottom, vmul(f1dr, top));
    if constexpr (CLIP) {
      // skimage keeps exact-cval (0) outputs when 0 lies outside the slice
      // range; an output is exactly 0 iff no in-range tap has positive weight.
      const bool colw = vc0 || (dc > 0.0 && vc1);
      const bool anyin = (vr0 && colw) || (dr > 0.0 && vr1 && colw);
      if (anyin) v = vclamp(v, lo, hi);
    }
    if (g.occ) {
      const float yr = (float)(r - g.c);
#pragma unroll
      for (int q = 0; q < ZV; ++q)
        if (yr > lim[q]) vset(v, q, 0.0f);
    }
    acc = vfma(abs_weight(g, t, (double)(r - g.c)), v, acc);
  }
  return acc;
}

// forward projection with inclination, one detector row j
__device__ __forceinline__ float fp_ray_incl(const ParDev& g, const float* __restrict__ vol, int k, int i, int j) {
  const int n = g.n, nz = g.nz;
  const double* M = g.mats + 6 * i;
  const double kp = (double)k - g.det_offset;
  const double a0 = M[0] * kp, a1 = M[3] * kp;
  const double t = (double)(k - g.c) - g.det_offset;
  float acc = 0.0f;
  for (int r = 0; r < n; ++r) {
    const double rr = (double)r;
    const double col = (a0 + M[1] * rr) + M[2];
    const double row = (a1 + M[4] * rr) + M[5];
    if (!(row > -1.0 && row < (double)n && col > -1.0 && col < (double)n)) continue;
    const double s = (double)(r - g.c);
    const double zpos = (double)j + s * g.tan_phi;
    const double fz = floor(zpos);
    const double wz1 = zpos - fz;
    const int z0 = (int)fz;
    const double fr = floor(row), fc = floor(col);
    const double dr = row - fr, dc = col - fc;
    const int r0 = (int)fr, c0 = (int)fc, r1 = (int)ceil(row), c1 = (int)ceil(col);
    const bool vr0 = r0 >= 0, vr1 = r1 < n, vc0 = c0 >= 0, vc1 = c1 < n;
    const float f1dc = (float)(1.0 - dc), fdc = (float)dc;
    const float f1dr = (float)(1.0 - dr), fdr = (float)dr;
    float v = 0.0f;
    for (int q = 0; q < 2; ++q) {
      const int zz = z0 + q;
      if (zz < 0 || zz >= nz) continue;
      const float wz = (float)(q == 0 ? 1.0 - wz1 : wz1);
      float tl = 0.f, tr = 0.f, bl = 0.f, br = 0.f;
      if (vr0 && vc0) tl = vol[((size_t)r0 * n + c0) * nz + zz];
      if (vr0 && vc1) tr = vol[((size_t)r0 * n + c1) * nz + zz];
      if (vr1 && vc0) bl = vol[((size_t)r1 * n + c0) * nz + zz];
      if (vr1 && vc1) br = vol[((size_t)r1 * n + c1) * nz + zz];
      const float top = __builtin_fmaf(fdc, tr, f1dc * tl);
      const float bottom = __builtin_fmaf(fdc, br, f1dc * bl);
      v = __builtin_fmaf(wz, __builtin_fmaf(fdr, bottom, f1dr * top), v);
    }
    acc = __builtin_fmaf(abs_weight(g, t, s), v, acc);
  }
  return acc;
}

// ---------------------------------------------------------------------------
// back projection at voxel column pix, z .. z+ZV-1 (no circle clip here)
// (Projector3DParallel.py:175-205)
// ---------------------------------------------------------------------------
// Occlusion of a voxel at detector coordinate t, along-ray coordinate s,
// for angle i and slices z..z+ZV-1: the voxel gets nothing from this angle
// when s > floor(np.interp(t, xp, occ column, left=nan, right=nan))
// (Projector3DParallel.py:192-199, 209-216).  np.interp returns fp[j]
// exactly when t equals a node xp[j] (also the last one) and otherwise
// evaluates slope * (t - xp[j]) + fp[j] on the interval containing t (NaN if
// a node is NaN); NaN compares false.  t is inside [xp[0], xp[n-1]] here
// (interp_node accepted it).
template <int ZV>
__device__ __forceinline__ void occ_shadow_mask(const ParDev& g, int i, int j, double t, double s, int z,
                                                typename VecT<ZV>::T& val) {
  const size_t zs = (size_t)g.nz;
  const float* oc = g.occ + (size_t)i * zs + z;
  const size_t step_j = (size_t)g.na * zs;
  // numpy's interval: xp[jn] <= t < xp[jn + 1], found by comparing t with
  // the node values (floor(t - xp[0]) can be off by one when t is within an
  // ulp of a node)
  int jn = j;
  if (jn > 0 && t < (double)(jn - g.c) - g.det_offset) {
    --jn;
  } else if (jn < g.n - 1 && t >= (double)(jn + 1 - g.c) - g.det_offset) {
    ++jn;
  }
#pragma unroll
  for (int q = 0; q < ZV; ++q) {
    const double x0 = (double)(jn - g.c) - g.det_offset;
    const double o0 = (double)oc[(size_t)jn * step_j + q];
    double o = o0;
    if (jn < g.n - 1 && t != x0) {
      const double o1 = (double)oc[(size_t)(jn + 1) * step_j + q];
      const double x1 = (double)(jn + 1 - g.c) - g.det_offset;
      const double slope = (o1 - o0) / (x1 - x0);
      o = slope * (t - x0) + o0;
    }
    if (s > floor(o)) vset(val, q, 0.0f);
  }
}

template <int ZV>
__device__ __forceinline__ typename VecT<ZV>::T bp_voxel(const ParDev& g, const float* __restrict__ sino, int pix,
                                                          int z) {
  using V = typename VecT<ZV>::T;
  const int row = pix / g.n, col = pix % g.n;
  const double x = (double)(col - g.c), y = (double)(row - g.c);
  const size_t zstride = (size_t)g.nz;
  V acc = vzero<ZV>();
  for (int i = 0; i < g.na; ++i) {
    const double co = g.cs[2 * i], sn = g.cs[2 * i + 1];
    const double t = x * co - y * sn;
    int j, j1;
    float w;
    if (!interp_node(g, t, j, j1, w)) continue;
    const V b0 = vload<ZV>(sino + ((size_t)j * g.na + i) * zstride + z);
    const V b1 = vload<ZV>(sino + ((size_t)j1 * g.na + i) * zstride + z);
    V val = vfma(w, vsub(b1, b0), b0);
    if (g.mu != 0.0) val = vmul(abs_weight(g, t, x * sn + y * co), val);
    if (g.occ) occ_shadow_mask<ZV>(g, i, j, t, x * sn + y * co, z, val);
    acc = vadd(acc, val);
  }
  return acc;
}

__device__ __forceinline__ float bp_voxel_incl(const ParDev& g, const float* __restrict__ sino, int pix, int z) {
  const int row = pix / g.n, col = pix % g.n;
  const double x = (double)(col - g.c), y = (double)(row - g.c);
  float acc = 0.0f;
  for (int i = 0; i < g.na; ++i) {
    const double co = g.cs[2 * i], sn = g.cs[2 * i + 1];
    const double t = x * co - y * sn;
    int j, j1;
    float w;
    if (!interp_node(g, t, j, j1, w)) continue;
    const double s = x * sn + y * co;
    const double vpos = (double)z - s * g.tan_phi;
    const double fz = floor(vpos);
    const double wz1 = vpos - fz;
    const int q0 = (int)fz;
    float val = 0.0f;
    for (int q = 0; q < 2; ++q) {
      const int jz = q0 + q;
      if (jz < 0 || jz >= g.nz) continue;
      const float wz = (float)(q == 0 ? 1.0 - wz1 : wz1);
      const float b0 = sino[((size_t)j * g.na + i) * g.nz + jz];
      const float b1 = sino[((size_t)j1 * g.na + i) * g.nz + jz];
      val = __builtin_fmaf(wz, __builtin_fmaf(w, b1 - b0, b0), val);
    }
    acc = __builtin_fmaf(abs_weight(g, t, s), val, acc);
  }
  return acc;
}

// ---------------------------------------------------------------------------
// exact transpose of the forward projection (linear part): voxel-driven
// gather over the <= 4x4 candidate samples (k, r) per angle whose bilinear
// footprint covers the voxel
// ---------------------------------------------------------------------------
template <int ZV>
__device__ __forceinline__ typename VecT<ZV>::T fpT_voxel(const ParDev& g, const float* __restrict__ sino, int pix,
                                                           int z) {
  using V = typename VecT<ZV>::T;
  const int n = g.n;
  const int row = pix / n, col = pix % n;
  const double X = (double)(col - g.c), Y = (double)(row - g.c);
  const size_t zstride = (size_t)g.nz;
  V acc = vzero<ZV>();
  for (int i = 0; i < g.na; ++i) {
    const double* M = g.mats + 6 * i;
    const double co = M[0], sn = M[1];
    const double kstar = co * X - sn * Y + (double)g.c + g.det_offset;
    const double rstar = sn * X + co * Y + (double)g.c;
    const int kb = (int)floor(kstar) - 1, rb = (int)floor(rstar) - 1;
    for (int kk = kb; kk < kb + 4; ++kk) {
      if (kk < 0 || kk >= n) continue;
      const double kp = (double)kk - g.det_offset;
      const double a0 = M[0] * kp, a1 = M[3] * kp;
      const double t = (double)(kk - g.c) - g.det_offset;
      float wk = 0.0f;
      for (int r = rb; r < rb + 4; ++r) {
        if (r < 0 || r >= n) continue;
        const double rr = (double)r;
        const double colS = (a0 + M[1] * rr) + M[2];
        const double rowS = (a1 + M[4] * rr) + M[5];
        if (!(fabs(rowS - (double)row) < 1.0 && fabs(colS - (double)col) < 1.0)) continue;
        const float wr = tap_weight_axis(rowS, row);
        const float wc = tap_weight_axis(colS, col);
        wk = __builtin_fmaf(wr * wc, abs_weight(g, t, (double)(r - g.c)), wk);
      }
      if (wk != 0.0f) acc = vfma(wk, vload<ZV>(sino + ((size_t)kk * g.na + i) * zstride + z), acc);
    }
  }
  return acc;
}

__device__ __forceinline__ float fpT_voxel_incl(const ParDev& g, const float* __restrict__ sino, int pix, int z) {
  const int n = g.n, nz = g.nz;
  const int row = pix / n, col = pix % n;
  const double X = (double)(col - g.c), Y = (double)(row - g.c);
  float acc = 0.0f;
  for (int i = 0; i < g.na; ++i) {
    const double* M = g.mats + 6 * i;
    const double co = M[0], sn = M[1];
    const double kstar = co * X - sn * Y + (double)g.c + g.det_offset;
    const double rstar = sn * X + co * Y + (double)g.c;
    const int kb = (int)floor(kstar) - 1, rb = (int)floor(rstar) - 1;
    for (int kk = kb; kk < kb + 4; ++kk) {
      if (kk < 0 || kk >= n) continue;
      const double kp = (double)kk - g.det_offset;
      const double a0 = M[0] * kp, a1 = M[3] * kp;
      const double t = (double)(kk - g.c) - g.det_offset;
      for (int r = rb; r < rb + 4; ++r) {
        if (r < 0 || r >= n) continue;
        const double rr = (double)r;
        const double colS = (a0 + M[1] * rr) + M[2];
        const double rowS = (a1 + M[4] * rr) + M[5];
        if (!(fabs(rowS - (double)row) < 1.0 && fabs(colS - (double)col) < 1.0)) continue;
        const float wxy = tap_weight_axis(rowS, row) * tap_weight_axis(colS, col);
        if (wxy == 0.0f) continue;
        const double s = (double)(r - g.c);
        const float wa = abs_weight(g, t, s) * wxy;
        // detector rows j whose sample z position j + s tan(phi) has a tap on z
        const int jc = (int)floor((double)z - s * g.tan_phi);
        for (int j = jc - 1; j <= jc + 2; ++j) {
          if (j < 0 || j >= nz) continue;
          const float wz = tap_weight_axis((double)j + s * g.tan_phi, z);
          if (wz == 0.0f) continue;
          acc = __builtin_fmaf(wa * wz, sino[((size_t)kk * g.na + i) * nz + j], acc);
        }
      }
    }
  }
  return acc;
}

// ---------------------------------------------------------------------------
// exact transpose of the back projection: sinogram-driven gather over the
// voxels whose detector coordinate lies within one bin of bin k
// ---------------------------------------------------------------------------
__device__ __forceinline__ void bpT_range(const ParDev& g, double co, double sn, double xk, int a, bool rows_major,
                                          int& b0, int& b1) {
  double lo, hi;
  if (rows_major) {
    const double Y = (double)(a - g.c);
    const double e0 = (xk - 1.0 + Y * sn) / co, e1 = (xk + 1.0 + Y * sn) / co;
    lo = fmin(e0, e1);
    hi = fmax(e0, e1);
  } else {
    const double X = (double)(a - g.c);
    const double e0 = (X * co - (xk - 1.0)) / sn, e1 = (X * co - (xk + 1.0)) / sn;
    lo = fmin(e0, e1);
    hi = fmax(e0, e1);
  }
  b0 = (int)floor(lo) - 1 + g.c;
  b1 = (int)ceil(hi) + 1 + g.c;
  if (b0 < 0) b0 = 0;
  if (b1 > g.n - 1) b1 = g.n - 1;
}

template <int ZV>
__device__ __forceinline__ typename VecT<ZV>::T bpT_bin(const ParDev& g, const float* __restrict__ vol, int k, int i,
                                                         int z, int clipc) {
  using V = typename VecT<ZV>::T;
  const int n = g.n;
  const size_t zstride = (size_t)g.nz;
  const double co = g.cs[2 * i], sn = g.cs[2 * i + 1];
  const double xk = (double)(k - g.c) - g.det_offset;
  const bool rows_major = fabs(co) >= fabs(sn);
  V acc = vzero<ZV>();
  for (int a = 0; a < n; ++a) {
    int b0, b1;
    bpT_range(g, co, sn, xk, a, rows_major, b0, b1);
    for (int bb = b0; bb <= b1; ++bb) {
      const int row = rows_major ? a : bb;
      const int col = rows_major ? bb : a;
      const int pix = row * n + col;
      if (clipc && g.outside[pix]) continue;
      const double x = (double)(col - g.c), y = (double)(row - g.c);
      const double t = x * co - y * sn;
      int j, j1;
      float w;
      if (!interp_node(g, t, j, j1, w)) continue;
      float wk = 0.0f;
      if (j == k) wk += 1.0f - w;
      if (j1 == k) wk += w;
      if (wk == 0.0f) continue;
      if (g.mu != 0.0) wk *= abs_weight(g, t, x * sn + y * co);
      acc = vfma(wk, vload<ZV>(vol + (size_t)pix * zstride + z), acc);
    }
  }
  return acc;
}

__device__ __forceinline__ float bpT_bin_incl(const ParDev& g, const float* __restrict__ vol, int k, int i, int jz,
                                              int clipc) {
  const int n = g.n, nz = g.nz;
  const double co = g.cs[2 * i], sn = g.cs[2 * i + 1];
  const double xk = (double)(k - g.c) - g.det_offset;
  const bool rows_major = fabs(co) >= fabs(sn);
  float acc = 0.0f;
  for (int a = 0; a < n; ++a) {
    int b0, b1;
    bpT_range(g, co, sn, xk, a, rows_major, b0, b1);
    for (int bb = b0; bb <= b1; ++bb) {
      const int row = rows_major ? a : bb;
      const int col = rows_major ? bb : a;
      const int pix = row * n + col;
      if (clipc && g.outside[pix]) continue;
      const double x = (double)(col - g.c), y = (double)(row - g.c);
      const double t = x * co - y * sn;
      int j, j1;
      float w;
      if (!interp_node(g, t, j, j1, w)) continue;
      float wk = 0.0f;
      if (j == k) wk += 1.0f - w;
      if (j1 == k) wk += w;
      if (wk == 0.0f) continue;
      const double s = x * sn + y * co;
      wk *= abs_weight(g, t, s);
      // voxels z whose detector-row position z - s tan(phi) has a tap on jz
      const int zc = (int)floor((double)jz + s * g.tan_phi);
      for (int z = zc - 1; z <= zc + 2; ++z) {
        if (z < 0 || z >= nz) continue;
        const float wz = tap_weight_axis((double)z - s * g.tan_phi, jz);
        if (wz == 0.0f) continue;
        acc = __builtin_fmaf(wk * wz, vol[(size_t)pix * nz + z], acc);
      }
    }
  }
  return acc;
}


// ---------------------------------------------------------------------------
// wavefront-uniform cores
//
// When a wavefront's 64 lanes cover 64*ZV consecutive z values of ONE ray (or
// voxel column), the geometry of a sample (or angle) is the same for every
// lane.  Lane l then evaluates the geometry of sample r0 + l (or angle
// i0 + l) -- 64 samples in parallel, float64, the reference's operation order
// -- and the inner loop walks the samples with an in-range tap (a ballot
// mask), broadcasting each sample's tap base and weights with readlane into
// scalar registers: per sample the vector units only issue the tap loads and
// the fused multiply-adds.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int rl_i(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// ---------------------------------------------------------------------------
// Exact transposes, wavefront-uniform (zero inclination).  A wavefront owns
// one detector bin (B^T) or one voxel column (A^T) and 64*ZV consecutive z.
// Lane l evaluates, in float64 and with exactly the per-lane cores'
// arithmetic, the taps of row a0 + l of the bin's strip (B^T) or of angle
// i0 + l (A^T): at most four (voxel or detector bin, weight) pairs with a
// nonzero weight, in the per-lane cores' order.  They pass through a
// per-wavefront LDS buffer; the wave then walks the rows (angles) in order
// with one coalesced load per tap, so each z sums the same terms in the same
// order as bpT_bin / fpT_voxel: the results are bitwise equal.
// ---------------------------------------------------------------------------
struct AdjSlot {
  float4* w;   // [64] tap weights (0 = no tap)
  int4* o;     // [64] tap voxel column (B^T) or sinogram row (A^T), -1 = none
};
__device__ __forceinline__ AdjSlot adj_lds_slot() {
  __shared__ float4 w[4][64];
  __shared__ int4 o[4][64];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 3;
  return {w[wv], o[wv]};
}

__device__ __forceinline__ void adj_put(float4& w, int4& o, int m, float wk, int off) {
  if (m == 0) { w.x = wk; o.x = off; }
  else if (m == 1) { w.y = wk; o.y = off; }
  else if (m == 2) { w.z = wk; o.z = off; }
  else { w.w = wk; o.w = off; }
}

__device__ __forceinline__ void adj_putw(float4& w, int m, float wk) {
  if (m == 0) w.x = wk;
  else if (m == 1) w.y = wk;
  else if (m == 2) w.z = wk;
  else w.w = wk;
}

template <int ZV>
__device__ __forceinline__ typename VecT<ZV>::T adj_taps(const float* __restrict__ base, size_t stride, int zl,
                                                         const AdjSlot& sl, int rows, typename VecT<ZV>::T acc) {
  for (int r = 0; r < rows; ++r) {
    const float4 w = sl.w[r];
    const int4 o = sl.o[r];
    const int o0 = __builtin_amdgcn_readfirstlane(o.x), o1 = __builtin_amdgcn_readfirstlane(o.y);
    const int o2 = __builtin_amdgcn_readfirstlane(o.z), o3 = __builtin_amdgcn_readfirstlane(o.w);
    if (o0 >= 0) acc = vfma(w.x, vload<ZV>(base + (size_t)o0 * stride + zl), acc);
    if (o1 >= 0) acc = vfma(w.y, vload<ZV>(base + (size_t)o1 * stride + zl), acc);
    if (o2 >= 0) acc = vfma(w.z, vload<ZV>(base + (size_t)o2 * stride + zl), acc);
    if (o3 >= 0) acc = vfma(w.w, vload<ZV>(base + (size_t)o3 * stride + zl), acc);
  }
  return acc;
}

// B^T of bin (k, i): the voxels of each row (column, when |sin| > |cos|) of
// the strip |t - t_k| < 1, rows in order (bpT_bin)
template <int ZV>
__device__ __forceinline__ typename VecT<ZV>::T bpT_bin_wave(const ParDev& g, const float* __restrict__ vol, int k,
                                                              int i, int zl, int lane, int clipc) {
  using V = typename VecT<ZV>::T;
  const int n = g.n;
  const double co = g.cs[2 * i], sn = g.cs[2 * i + 1];
  const double xk = (double)(k - g.c) - g.det_offset;
  const bool rows_major = fabs(co) >= fabs(sn);
  const AdjSlot sl = adj_lds_slot();
  V acc = vzero<ZV>();
  for (int a0 = 0; a0 < n; a0 += 64) {
    const int a = a0 + lane;
    float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
    int4 o = make_int4(-1, -1, -1, -1);
    if (a < n) {
      int b0, b1;
      bpT_range(g, co, sn, xk, a, rows_major, b0, b1);
      int m = 0;
      for (int bb = b0; bb <= b1 && m < 4; ++bb) {
        const int row = rows_major ? a : bb;
        const int col = rows_major ? bb : a;
        const int pix = row * n + col;
        if (clipc && g.outside[pix]) continue;
        const double x = (double)(col - g.c), y = (double)(row - g.c);
        const double t = x * co - y * sn;
        int j, j1;
        float wj;
        if (!interp_node(g, t, j, j1, wj)) continue;
        float wk = 0.0f;
        if (j == k) wk += 1.0f - wj;
        if (j1 == k) wk += wj;
        if (wk == 0.0f) continue;
        if (g.mu != 0.0) wk *= abs_weight(g, t, x * sn + y * co);
        adj_put(w, o, m, wk, pix);
        ++m;
      }
    }
    __builtin_amdgcn_wave_barrier();
    sl.w[lane] = w;
    sl.o[lane] = o;
    __builtin_amdgcn_wave_barrier();
    acc = adj_taps<ZV>(vol, (size_t)g.nz, zl, sl, n - a0 < 64 ? n - a0 : 64, acc);
  }
  return acc;
}

// weight of voxel (x, y) in B^T of bin k at the angle (co, sn): bpT_bin's
// arithmetic, 0 when the voxel is outside the bin's strip
__device__ __forceinline__ float bpT_weight(const ParDev& g, double co, double sn, int k, double x, double y) {
  const double t = x * co - y * sn;
  int j, j1;
  float wj;
  if (!interp_node(g, t, j, j1, wj)) return 0.0f;
  float wk = 0.0f;
  if (j == k) wk += 1.0f - wj;
  if (j1 == k) wk += wj;
  if (wk == 0.0f) return 0.0f;
  if (g.mu != 0.0) wk *= abs_weight(g, t, x * sn + y * co);
  return wk;
}

// B^T of bin (k, i) and of the opposite bin (k2, i2): angle i2 is angle
// i + 180 deg and k2 = 2c + 2 det_offset - k, so t2 = -t and the two strips
// hold the same voxels.  Each voxel column of the strip is loaded once and
// feeds both sums.  The partner's weights use its own angle's cos / sin; both
// sums walk the primary's rows (columns) in order, which is the partner's own
// order whenever the two angles agree on the row direction (all but exact
// 45-degree multiples), so each sum is bpT_bin_wave's to the bit there.  Per
// row the two strips have at most 3 voxels together (|t - t_k| < 1 on a row
// where t moves >= 1/sqrt(2) per voxel; the partner's strip differs by the
// pairing tolerance only), within the 4 slots.
struct AdjSlot2 {
  float4* w;   // [64] primary tap weights
  float4* w2;  // [64] partner tap weights
  int4* o;     // [64] tap voxel column, -1 = none
};
__device__ __forceinline__ AdjSlot2 adj_lds_slot2() {
  __shared__ float4 w[4][64];
  __shared__ float4 w2[4][64];
  __shared__ int4 o[4][64];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 3;
  return {w[wv], w2[wv], o[wv]};
}

template <int ZV>
__device__ __forceinline__ void bpT_pair_wave(const ParDev& g, const float* __restrict__ vol, int k, int i, int k2,
                                              int i2, int zl, int lane, int clipc, typename VecT<ZV>::T& acc,
                                              typename VecT<ZV>::T& acc2) {
  const int n = g.n;
  const size_t stride = (size_t)g.nz;
  const double co = g.cs[2 * i], sn = g.cs[2 * i + 1];
  const double co2 = g.cs[2 * i2], sn2 = g.cs[2 * i2 + 1];
  const double xk = (double)(k - g.c) - g.det_offset;
  const bool rows_major = fabs(co) >= fabs(sn);
  const AdjSlot2 sl = adj_lds_slot2();
  acc = vzero<ZV>();
  acc2 = vzero<ZV>();
  for (int a0 = 0; a0 < n; a0 += 64) {
    const int a = a0 + lane;
    float4 w = make_float4(0.f, 0.f, 0.f, 0.f), w2 = w;
    int4 o = make_int4(-1, -1, -1, -1);
    if (a < n) {
      int b0, b1;
      bpT_range(g, co, sn, xk, a, rows_major, b0, b1);
      int m = 0;
      for (int bb = b0; bb <= b1 && m < 4; ++bb) {
        const int row = rows_major ? a : bb;
        const int col = rows_major ? bb : a;
        const int pix = row * n + col;
        if (clipc && g.outside[pix]) continue;
        const double x = (double)(col - g.c), y = (double)(row - g.c);
        const float wk = bpT_weight(g, co, sn, k, x, y);
        const float wk2 = bpT_weight(g, co2, sn2, k2, x, y);
        if (wk == 0.0f && wk2 == 0.0f) continue;
        adj_put(w, o, m, wk, pix);
        adj_putw(w2, m, wk2);
        ++m;
      }
    }
    __builtin_amdgcn_wave_barrier();
    sl.w[lane] = w;
    sl.w2[lane] = w2;
    sl.o[lane] = o;
    __builtin_amdgcn_wave_barrier();
    const int rows = n - a0 < 64 ? n - a0 : 64;
    for (int r = 0; r < rows; ++r) {
      const float4 wr = sl.w[r], wr2 = sl.w2[r];
      const int4 orr = sl.o[r];
      const int o0 = __builtin_amdgcn_readfirstlane(orr.x), o1 = __builtin_amdgcn_readfirstlane(orr.y);
      const int o2 = __builtin_amdgcn_readfirstlane(orr.z), o3 = __builtin_amdgcn_readfirstlane(orr.w);
      if (o0 >= 0) {
        const typename VecT<ZV>::T v = vload<ZV>(vol + (size_t)o0 * stride + zl);
        acc = vfma(wr.x, v, acc);
        acc2 = vfma(wr2.x, v, acc2);
      }
      if (o1 >= 0) {
        const typename VecT<ZV>::T v = vload<ZV>(vol + (size_t)o1 * stride + zl);
        acc = vfma(wr.y, v, acc);
        acc2 = vfma(wr2.y, v, acc2);
      }
      if (o2 >= 0) {
        const typename VecT<ZV>::T v = vload<ZV>(vol + (size_t)o2 * stride + zl);
        acc = vfma(wr.z, v, acc);
        acc2 = vfma(wr2.z, v, acc2);
      }
      if (o3 >= 0) {
        const typename VecT<ZV>::T v = vload<ZV>(vol + (size_t)o3 * stride + zl);
        acc = vfma(wr.w, v, acc);
        acc2 = vfma(wr2.w, v, acc2);
      }
    }
  }
}

// A^T of voxel column pix: the detector bins of each angle whose samples
// tap the voxel, angles in order (fpT_voxel)
template <int ZV>
__device__ __forceinline__ typename VecT<ZV>::T fpT_voxel_wave(const ParDev& g, const float* __restrict__ sino,
                                                                int pix, int zl, int lane) {
  using V = typename VecT<ZV>::T;
  const int n = g.n;
  const int row = pix / n, col = pix % n;
  const double X = (double)(col - g.c), Y = (double)(row - g.c);
  const AdjSlot sl = adj_lds_slot();
  V acc = vzero<ZV>();
  for (int i0 = 0; i0 < g.na; i0 += 64) {
    const int i = i0 + lane;
    float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
    int4 o = make_int4(-1, -1, -1, -1);
    if (i < g.na) {
      const double* M = g.mats + 6 * i;
      const double co = M[0], sn = M[1];
      const double kstar = co * X - sn * Y + (double)g.c + g.det_offset;
      const double rstar = sn * X + co * Y + (double)g.c;
      const int kb = (int)floor(kstar) - 1, rb = (int)floor(rstar) - 1;
      int m = 0;
      for (int kk = kb; kk < kb + 4; ++kk) {
        if (kk < 0 || kk >= n) continue;
        const double kp = (double)kk - g.det_offset;
        const double a0 = M[0] * kp, a1 = M[3] * kp;
        const double t = (double)(kk - g.c) - g.det_offset;
        float wk = 0.0f;
        for (int r = rb; r < rb + 4; ++r) {
          if (r < 0 || r >= n) continue;
          const double rr = (double)r;
          const double colS = (a0 + M[1] * rr) + M[2];
          const double rowS = (a1 + M[4] * rr) + M[5];
          if (!(fabs(rowS - (double)row) < 1.0 && fabs(colS - (double)col) < 1.0)) continue;
          const float wr = tap_weight_axis(rowS, row);
          const float wc = tap_weight_axis(colS, col);
          wk = __builtin_fmaf(wr * wc, abs_weight(g, t, (double)(r - g.c)), wk);
        }
        if (wk != 0.0f) {
          adj_put(w, o, m, wk, kk * g.na + i);
          ++m;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
    sl.w[lane] = w;
    sl.o[lane] = o;
    __builtin_amdgcn_wave_barrier();
    acc = adj_taps<ZV>(sino, (size_t)g.nz, zl, sl, g.na - i0 < 64 ? g.na - i0 : 64, acc);
  }
  return acc;
}

// the transposes' lanes own ZV consecutive slices: those past nz load a copy of
// the last ones and store nothing
template <int ZV>
__device__ __forceinline__ int wave_zload(int z, int nz) { return z < nz - ZV ? z : nz - ZV; }
template <int ZV>
__device__ __forceinline__ void wave_zstore(float* col, int z, int nz, typename VecT<ZV>::T v) {
  if (z < nz) vstore<ZV>(col + z, v);
}

// Slices of a lane in the forward's wavefronts: ZV consecutive ones, or (SPLIT)
// z + 64 q, q < ZV, with a 4-byte load each.  Lanes past nz load a copy of the
// last valid slices and store nothing.
template <int ZV, bool SPLIT>
struct FpLane {
  using V = typename VecT<ZV>::T;
  int z;
  uint32_t zb[SPLIT ? ZV : 1];   // byte offsets of the loads
  __device__ __forceinline__ FpLane(int chunk, int lane, int nz) {
    z = chunk * 64 * ZV + (SPLIT ? lane : lane * ZV);
    if constexpr (SPLIT) {
#pragma unroll
      for (int q = 0; q < ZV; ++q) zb[q] = 4u * (uint32_t)(z + 64 * q < nz - 1 ? z + 64 * q : nz - 1);
    } else {
      zb[0] = 4u * (uint32_t)(z < nz - ZV ? z : nz - ZV);
    }
  }
  __device__ __forceinline__ V load(__amdgpu_buffer_rsrc_t r, uint32_t soff) const {
    if constexpr (SPLIT) {
      V v;
#pragma unroll
      for (int q = 0; q < ZV; ++q) vset(v, q, bload<1>(r, zb[q], soff));
      return v;
    } else {
      return bload<ZV>(r, zb[0], soff);
    }
  }
  // the lane's values of an array over z
  __device__ __forceinline__ V values(const float* __restrict__ a) const {
    if constexpr (SPLIT) {
      V v;
#pragma unroll
      for (int q = 0; q < ZV; ++q) vset(v, q, a[zb[q] / 4]);
      return v;
    } else {
      return vload<ZV>(a + zb[0] / 4);
    }
  }
  __device__ __forceinline__ void store(float* col, int nz, V v) const {
    if constexpr (SPLIT) {
#pragma unroll
      for (int q = 0; q < ZV; ++q)
        if (z + 64 * q < nz) col[z + 64 * q] = vget(v, q);
    } else {
      if (z < nz) vstore<ZV>(col + z, v);
    }
  }
};

// The warp clip of a slice is a no-op when 0 lies in [min, max] of the slice:
// bilinear samples are convex combinations of the slice's values and the zero
// padding.  Whether it is not one for any of the wavefront's slices (lo, hi: their
// least and largest values).
template <int ZV>
__device__ __forceinline__ bool wave_clip_active(const typename VecT<ZV>::T& lo, const typename VecT<ZV>::T& hi) {
  bool need = false;
#pragma unroll
  for (int q = 0; q < ZV; ++q) need |= !(vget(lo, q) <= 0.0f && 0.0f <= vget(hi, q));
  return __ballot(need) != 0ull;
}
template <int ZV, bool SPLIT>
__device__ __forceinline__ bool wave_clip_active(const float* __restrict__ minmax, int nz, const FpLane<ZV, SPLIT>& ln) {
  return wave_clip_active<ZV>(ln.values(minmax), ln.values(minmax + nz));
}

// slot weights of one axis: the taps floor / floor+1 (skimage's floor / ceil
// with weights 1-d / d) mapped onto the pair (b, b+1) with b in [0, n-2]
__device__ __forceinline__ void axis_slots(double coord, int n, int& b, double& s0, double& s1) {
  const double f = floor(coord);
  const double d = coord - f;
  const int fi = (int)f;
  if (fi < 0) {          // floor = -1: only floor+1 = 0 is a tap
    b = 0; s0 = d; s1 = 0.0;
  } else if (fi >= n - 1) {  // floor = n-1: floor+1 = n is outside
    b = n - 2; s0 = 0.0; s1 = 1.0 - d;
  } else {
    b = fi; s0 = 1.0 - d; s1 = d;
  }
}

// forward projection of ray (k, i), lanes = z; requires n >= 2.  REUSE keeps
// the previous sample's four taps in registers: between consecutive samples
// the floor corner b moves by at most one pixel per axis, and when it moves
// along one axis only, two of the four taps are the previous sample's.  b is
// wave-uniform, so the case test is a scalar branch.  Lanes evaluate the
// geometry of 64 samples at once; the per-sample loop takes the cell from
// the sample's lane and its weights from the LDS buffer (fp_lds_slot).
//
// PAIR also projects the opposite ray, k2 = 2c + D - k at angle i + 180 deg,
// into *acc2: its sample r2 lies on sample r = 2c - r2 of ray k (rotating by
// 180 deg negates the matrix's linear part, and D = 2 det_offset maps the
// detector coordinate t to -t), so the taps are loaded once and weighted
// twice.  Ray k's samples are r = 0..n-1, the partner's r = 2c-n+1..2c; the
// loop runs over their union, each ray weighting only its own samples (the
// other's extra end sample adds an exact zero).  Each sample is interpolated
// once and multiplied by each ray's absorption weight (unpaired, the weight
// folds into the taps' weights: the sums agree to float32 rounding).  The
// partner's samples are summed in reverse order, at positions computed from
// angle i's matrix -- equal to the partner's own to ~1e-13 pixel, which moves
// the result by as little since the unclipped sample is continuous in its
// position.  The warp clip is not: a sample a
// rounding error inside the -1 or n border clips up to the slice minimum
// while one on the border stays 0, so PAIR excludes CLIP and clipped waves
// project the two rays separately.
// Per-wavefront LDS buffers through which the wavefront cores hand each
// lane's sample weights to the whole wavefront: a broadcast LDS read per
// sample replaces one cross-lane move per weight.  One buffer per kernel
// (these functions are not templates), for blocks of at most 4 wavefronts.
struct FpSlot {
  float4* w;   // [64] the four bilinear tap weights of each lane's sample
  float2* a;   // [64] its absorption weights (ray, partner ray)
};
__device__ __forceinline__ FpSlot fp_lds_slot() {
  __shared__ float4 w[4][64];
  __shared__ float2 a[4][64];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 3;
  return {w[wv], a[wv]};
}

template <bool CLIP, bool REUSE, bool PAIR, int ZV, bool SPLIT>
__device__ __forceinline__ typename VecT<ZV>::T fp_ray_wave(const ParDev& g, const float* __restrict__ vol,
                                                             const float* __restrict__ minmax, int k, int i,
                                                             const FpLane<ZV, SPLIT>& ln, int lane,
                                                             typename VecT<ZV>::T* acc2 = nullptr) {
  using V = typename VecT<ZV>::T;
  static_assert(!(PAIR && CLIP), "the clipped sample is discontinuous at the border: no pairing");
  const int n = g.n;
  const double* M = g.mats + 6 * i;
  const double M01 = M[1], M02 = M[2], M11 = M[4], M12 = M[5];
  const double kp = (double)k - g.det_offset;
  const double a0 = M[0] * kp, a1 = M[3] * kp;
  const double t = (double)(k - g.c) - g.det_offset;
  V lo = vzero<ZV>(), hi = vzero<ZV>();
  if constexpr (CLIP) {
    lo = ln.values(minmax);
    hi = ln.values(minmax + g.nz);
  }
  const size_t nzs = (size_t)g.nz;
  const size_t step_c = nzs, step_r = (size_t)n * nzs;
  // taps are buffer loads: lane byte offset 4z, scalar byte offset of the voxel
  // column from the first row that the 64 samples reach (their rows span at most
  // 66; where 66 rows pass 32 bits, from the sample's own cell)
  const uint32_t oc = (uint32_t)(4 * step_c), orr = (uint32_t)(4 * step_r);
  const bool big = 66ull * orr + 4ull * nzs >= 0xffffffffull;
  V acc = vzero<ZV>(), accp = vzero<ZV>();
  // Tap registers by absolute parity: T<a><b> holds the tap of the current
  // cell whose volume row is even (a = 0) or odd (a = 1) and whose column is
  // even (b = 0) or odd (b = 1).  When the cell moves by one row or column
  // the taps it keeps stay where they are and the new ones replace exactly
  // the ones that left (same parity), so the window never shifts between
  // registers.  Each lane delivers, in that parity order, its sample's weights,
  // the taps' byte offsets and which of the four the sample before it lacked:
  // a sample tests four bits and moves one offset from its lane per new tap.
  // (The scalar unit, one instruction per cycle for a CU's four SIMDs, was what
  // bound the loop when it found the case of 36 by comparing cell numbers and
  // built a descriptor per sample: 40 scalar instructions and branches.)
  V T00 = vzero<ZV>(), T01 = vzero<ZV>(), T10 = vzero<ZV>(), T11 = vzero<ZV>();
  const FpSlot sl = fp_lds_slot();
  bool number = true;   // one slice per lane: no sample was a NaN before the clip
  int last = -1;   // cell of the sample before the 64 (-1: none)
  const int r_end = PAIR ? (2 * g.c + 1 > n ? 2 * g.c + 1 : n) : n;
  const int r2_lo = 2 * g.c - n + 1;   // partner's first sample (PAIR)
  for (int r0 = 0; r0 < r_end; r0 += 64) {
    const int r = r0 + lane;
    int br = 0, bc = 0;
    float w00 = 0.f, w01 = 0.f, w10 = 0.f, w11 = 0.f, aw = 0.f;
    float aw2 = 0.f;
    bool valid = false, anyin = false;
    if (r < r_end) {
      const double rr = (double)r;
      const double col = (a0 + M01 * rr) + M02;
      const double row = (a1 + M11 * rr) + M12;
      if (row > -1.0 && row < (double)n && col > -1.0 && col < (double)n) {
        double r0w, r1w, c0w, c1w;
        axis_slots(row, n, br, r0w, r1w);
        axis_slots(col, n, bc, c0w, c1w);
        anyin = (r0w > 0.0 || r1w > 0.0) && (c0w > 0.0 || c1w > 0.0);
        if (!PAIR || r < n) aw = abs_weight(g, t, (double)(r - g.c));
        if constexpr (PAIR) {
          if (r >= r2_lo) aw2 = abs_weight(g, -t, (double)(g.c - r));
        }
        valid = anyin && (CLIP || aw != 0.0f || aw2 != 0.0f);
        // unpaired without the clip, the absorption folds into the weights;
        // paired, the sample is interpolated once and weighted per ray
        const float f = (CLIP || PAIR) ? 1.0f : aw;
        const float k00 = f * (float)(r0w * c0w), k01 = f * (float)(r0w * c1w);
        const float k10 = f * (float)(r1w * c0w), k11 = f * (float)(r1w * c1w);
        // parity (a, b) holds corner (a ^ row parity, b ^ column parity)
        const bool pr = br & 1, pc = bc & 1;
        const float e0 = pc ? k01 : k00, e1 = pc ? k00 : k01;   // row 0 by column parity
        const float f0 = pc ? k11 : k10, f1 = pc ? k10 : k11;   // row 1
        w00 = pr ? f0 : e0;
        w01 = pr ? f1 : e1;
        w10 = pr ? e0 : f0;
        w11 = pr ? e1 : f1;
      }
    }
    unsigned long long m = __ballot(valid);
    if (!m) {
      last = -1;
      continue;
    }
    // taps that the sample before (in the lane before) does not hold
    const int cell = valid ? (br << 14) | bc : -1;   // n < 2^14
    const int up = __shfl_up(cell, 1), before = lane == 0 ? last : up;
    last = rl_i(cell, 63);
    const int dr = br - (before >> 14), dc = bc - (before & 0x3fff);
    int lacks = 15;   // bit 2 a + b: the tap of row parity a, column parity b
    if (REUSE && before >= 0 && dr >= -1 && dr <= 1 && dc >= -1 && dc <= 1)
      lacks = (dr ? 3 << (2 * ((br + (dr > 0)) & 1)) : 0) | (dc ? 5 << ((bc + (dc > 0)) & 1) : 0);
    const int row_lo = min(rl_i(br, __builtin_ctzll(m)), rl_i(br, 63 - __builtin_clzll(m)));
    const uint32_t at = big ? 0u : (uint32_t)(br - row_lo) * orr + (uint32_t)bc * oc;
    // the tap of parity (a, b) is the corner (a ^ row parity, b ^ column parity)
    const uint32_t re = at + ((br & 1) ? orr : 0u), ro = at + ((br & 1) ? 0u : orr);
    const uint32_t ce = (bc & 1) ? oc : 0u, co = (bc & 1) ? 0u : oc;
    const int a00 = (int)(re + ce), a01 = (int)(re + co), a10 = (int)(ro + ce), a11 = (int)(ro + co);
    __amdgpu_buffer_rsrc_t rs = buf_rsrc(vol + (size_t)row_lo * step_r, 0xffffffffu);
    // the wave's previous reads of the buffers precede these writes (LDS
    // operations of a wavefront complete in order)
    __builtin_amdgcn_wave_barrier();
    sl.w[lane] = make_float4(w00, w01, w10, w11);
    sl.a[lane] = make_float2(aw, aw2);
    __builtin_amdgcn_wave_barrier();
    // Unpaired without the clip (absorption in the taps' weights) the samples are
    // summed 16 at a time: the whole ray's sum is rounded once per 16 samples
    constexpr int kPart = CLIP || PAIR ? 64 : 16;
#pragma unroll 1
    for (int from = 0; from < 64; from += kPart) {
      unsigned long long ms = kPart < 64 ? m & (0xffffull << from) : m;
      V part = vzero<ZV>();
      while (ms) {
        const int j = __builtin_ctzll(ms);
        ms &= ms - 1;
        const float4 Q = sl.w[j];
        const float q00 = Q.x, q01 = Q.y, q10 = Q.z, q11 = Q.w;
        const int load = rl_i(lacks, j);
        if (big) {
          const int at_j = rl_i(cell, j);
          rs = buf_rsrc(vol + (size_t)(at_j >> 14) * step_r + (size_t)(at_j & 0x3fff) * step_c, 0xffffffffu);
        }
        if (load & 1) T00 = ln.load(rs, (uint32_t)rl_i(a00, j));
        if (load & 2) T01 = ln.load(rs, (uint32_t)rl_i(a01, j));
        if (load & 4) T10 = ln.load(rs, (uint32_t)rl_i(a10, j));
        if (load & 8) T11 = ln.load(rs, (uint32_t)rl_i(a11, j));
        if constexpr (CLIP) {
          V v = vfma(q11, T11, vfma(q10, T10, vfma(q01, T01, vmul(q00, T00))));
          if constexpr (ZV == 1) number = number && v == v;
          v = vclamp(v, lo, hi);  // every enumerated sample has an in-range tap of positive weight
          acc = vfma(sl.a[j].x, v, acc);
        } else if constexpr (PAIR) {
          const V v = vfma(q11, T11, vfma(q10, T10, vfma(q01, T01, vmul(q00, T00))));
          const float2 A = sl.a[j];
          acc = vfma(A.x, v, acc);
          accp = vfma(A.y, v, accp);
        } else {
          part = vadd(part, vfma(q11, T11, vfma(q10, T10, vfma(q01, T01, vmul(q00, T00)))));
        }
      }
      if constexpr (!CLIP && !PAIR) acc = vadd(acc, part);
    }
  }
  if constexpr (PAIR) *acc2 = accp;
  if constexpr (ZV == 1 && CLIP)
    if (!number) acc = __builtin_nanf("");   // for fp_ray_finish
  return acc;
}

// One slice per lane (up to 64 slices): a sum that is not finite is summed again as
// fp_ray does it.  The core above weights whole cells, and both rays of a pair, with
// weights that may be 0, and a voxel without a finite value would make NaNs of rays
// that pass beside it.  Problems of 32 to 56 slices came from fp_ray, where it does
// not; with more slices per lane, whose kernels never had this, it cost 1 us of a
// small call and 1 % of a large one.
template <int ZV, bool SPLIT>
__device__ __forceinline__ void fp_ray_finish(const ParDev& g, const float* __restrict__ vol,
                                              const float* __restrict__ minmax, bool clip, int k, int i,
                                              const FpLane<ZV, SPLIT>& ln, typename VecT<ZV>::T& acc) {
  if constexpr (ZV == 1) {
    const bool bad = !(fabsf(acc) <= 3.4028234664e38f) && ln.z < g.nz;
    if (__ballot(bad) == 0ull) return;
    if (bad) acc = clip ? fp_ray<1, true>(g, vol, minmax, k, i, ln.z) : fp_ray<1, false>(g, vol, minmax, k, i, ln.z);
  }
}

// Slices of a lane in the back projection's wavefronts: CONTIG (ZV = 4) z ..
// z + 3, else z + 64 q (4-byte loads: a wavefront's takes a CU's texture path 8.5
// cycles, a 16-byte one, for four times the slices, 17 to 20, an 8-byte one as
// long as that).  Slices past nz load a copy of the last one and are not stored.
template <int ZV, bool CONTIG>
struct ZLane {
  static_assert(!CONTIG || ZV == 4, "contiguous slices are 16-byte loads");
  int z;
  uint32_t zb[CONTIG ? 1 : ZV];   // byte offsets of the loads
  __device__ __forceinline__ ZLane(int chunk, int lane, int nz) {
    z = chunk * 64 * ZV + (CONTIG ? 4 * lane : lane);
    if constexpr (CONTIG) {
      zb[0] = 4u * (uint32_t)(z < nz - 4 ? z : nz - 4);
    } else {
#pragma unroll
      for (int q = 0; q < ZV; ++q) zb[q] = 4u * (uint32_t)(z + 64 * q < nz - 1 ? z + 64 * q : nz - 1);
    }
  }
  __device__ __forceinline__ int slice(int q) const { return CONTIG ? z + q : z + 64 * q; }
};
typedef float mf4 __attribute__((ext_vector_type(4)));

// the lane's ZV slices of a row
template <int ZV, bool CONTIG>
__device__ __forceinline__ void zload(__amdgpu_buffer_rsrc_t r, const ZLane<ZV, CONTIG>& ln, uint32_t soff,
                                      float (&t)[ZV]) {
  if constexpr (CONTIG) {
    const float4 v = bload<4>(r, ln.zb[0], soff);
    t[0] = v.x; t[1] = v.y; t[2] = v.z; t[3] = v.w;
  } else {
#pragma unroll
    for (int q = 0; q < ZV; ++q) t[q] = bload<1>(r, ln.zb[q], soff);
  }
}

// Back projection of a patch of 2 x 4 voxel columns on one wavefront, lanes = z:
// two 2 x 2 quads side by side.  Pixel p (0..3) of quad h is at row r0 + (p >> 1),
// column c0 + 2 h + (p & 1); bit 4 h + p of `active` says whether it is computed
// (in range and not circle-clipped).  Within one angle the patch's detector
// coordinates lie within 3 |cos| + |sin| <= 3.2 of each other, so its lower
// np.interp nodes span at most 5 rows and it reads at most 6.
//
// Each row loaded is multiplied into the four columns of a quad by one
// v_mfma_f32_4x4x1_16b_f32: 16 independent 4 x 1 x 4 products, of which block
// b holds the quad's four weights (one per lane of the block) and the row's
// slices of lanes 4 b .. 4 b + 3, so lane l accumulates its slice for all four
// columns.  It rounds like the four fused multiply-adds it replaces (checked
// bitwise), takes 8 to 10 cycles against their 18, and needs neither the
// weights in scalar registers nor a branch per column and row: a column that
// does not use a row has weight 0 there.  Adding 0 * row changes nothing
// unless the row holds an infinity or a NaN, which then makes a NaN:
// bp_patch_store recomputes those.  Each column thus sums
// fma(w1, b[j+1], fma(w0, b[j], acc)) in angle order.
//
// Lanes first evaluate the float64 geometry of 16 angles and leave each
// pixel's weights for the patch's rows in a per-wavefront LDS table; the
// per-angle loop reads its lanes' weights from there and takes the angle's
// first row and row count from a lane.
//
// COMB (no absorption): the angles are the plan's units (an angle and its
// opposite, or one angle), and the opposite angle's rows, mirrored, are added
// to the primary's as they are loaded: a column at detector coordinate t of
// angle a is at -t of angle a + 180 deg, where the mirrored bins (2c + 2
// det_offset - k) have the same neighbours and fractions.  np.interp is
// continuous inside the detector, so the primary's interval and fraction serve
// both; at the detector's ends, where it drops to 0, a column that only one of
// the two angles sees takes that angle's own rows in further passes.
//
// Bound by issuing: a 1 KiB row load takes a CU's texture path 17 to 20 cycles
// (a 256-byte one 8.5), its products 4 * 2 * 8.5 cycles of one SIMD, and the two
// overlap little: 256^3 x 360 angles takes 1.4 M cycles per CU, of them 0.83 M for
// the loads, 0.87 M for products and vector instructions, 0.3 M for scalar ones.
// With 16-byte loads the next angle's rows are loaded before this angle's products
// (0.62 against 0.70 ms); with 4-byte loads the second set of rows costs more
// wavefronts than it gains (256 x 256 x 128: 0.45 against 0.39 ms).
// Measured, four columns a wavefront with scalar weights and branches -> patches:
//   256 x 256 x 256, 360 angles, mu = 0.01   0.83 -> 0.64 ms
//   256 x 256 x 64, 360 angles               493 -> 230 us
//   201 x 201 x 77, 240 angles, mu = 0       284 -> 154 us
//   200 x 200 x 180, 240 angles              608 -> 237 us
//   160 x 160 x 120, 180 angles              136 -> 118 us
//   64 x 64 x 64, 180 angles                 67 -> 48 us
// Tried and slower at 256^3: 4 x 4 columns a wavefront (0.78 ms against 0.70: too
// few wavefronts for their shares to be even), 8 x 8 tiles of columns with the rows
// in LDS, a barrier per two angles (1.22) or per angle with these products (0.87).
// Requires n >= 2 and all 64 lanes.
constexpr int BP_QUADS = 2, BP_ROWS = 6;
__device__ __forceinline__ int bp_bit_row(int bit) { return (bit >> 1) & 1; }
__device__ __forceinline__ int bp_bit_col(int bit) { return 2 * (bit >> 2) + (bit & 1); }

// a wavefront's table, [16 angles][4 pixels][8 rows] of the quads' weights
constexpr int BP_TABLE = 16 * 4 * 8;

// rows first .. first + M - 1 of angle i (COMB, i2 >= 0: plus the mirrored
// rows of i2), multiplied into the patch with the angle's weights
template <int ZV, bool CONTIG, bool COMB, int M>
__device__ __forceinline__ void bp_rows(const ParDev& g, const float* __restrict__ sino, int first, int i, int i2,
                                        const ZLane<ZV, CONTIG>& ln, const float2* wa,
                                        mf4 (&acc)[BP_QUADS][ZV]) {
  const uint32_t row_b = 4u * (uint32_t)g.na * (uint32_t)g.nz, rows_b = (M - 1) * row_b + 4u * (uint32_t)g.nz;
  const uint32_t at = ((uint32_t)first * (uint32_t)g.na + (uint32_t)i) * (uint32_t)g.nz;
  const __amdgpu_buffer_rsrc_t rs = buf_rsrc(sino + (size_t)at, rows_b);
  float T[M][ZV];
#pragma unroll
  for (int k = 0; k < M; ++k) zload<ZV, CONTIG>(rs, ln, k * row_b, T[k]);
  if constexpr (COMB) {
    if (i2 >= 0) {
      const int last = 2 * g.c + g.pair_D - first - (M - 1);   // mirror of the last row
      const uint32_t at2 = ((uint32_t)last * (uint32_t)g.na + (uint32_t)i2) * (uint32_t)g.nz;
      const __amdgpu_buffer_rsrc_t rs2 = buf_rsrc(sino + (size_t)at2, rows_b);
      float O[M][ZV];
#pragma unroll
      for (int k = 0; k < M; ++k) zload<ZV, CONTIG>(rs2, ln, (M - 1 - k) * row_b, O[k]);
#pragma unroll
      for (int k = 0; k < M; ++k)
#pragma unroll
        for (int q = 0; q < ZV; ++q) T[k][q] += O[k][q];
    }
  }
#pragma unroll
  for (int k = 0; k < M; ++k) {
    const float2 w = wa[k];
#pragma unroll
    for (int h = 0; h < BP_QUADS; ++h)
#pragma unroll
      for (int q = 0; q < ZV; ++q)
        acc[h][q] = __builtin_amdgcn_mfma_f32_4x4x1f32(vget(w, h), T[k][q], acc[h][q], 0, 0, 0);
  }
}

template <int ZV, bool CONTIG, bool COMB>
__device__ __forceinline__ void bp_rows_of(const ParDev& g, const float* __restrict__ sino, int rows, int first, int i,
                                           int i2, const ZLane<ZV, CONTIG>& ln,
                                           const float2* wa,
                                           mf4 (&acc)[BP_QUADS][ZV]) {
  switch (rows) {   // wave-uniform; 0: no pixel of the patch is seen
    case 2: bp_rows<ZV, CONTIG, COMB, 2>(g, sino, first, i, i2, ln, wa, acc); break;
    case 3: bp_rows<ZV, CONTIG, COMB, 3>(g, sino, first, i, i2, ln, wa, acc); break;
    case 4: bp_rows<ZV, CONTIG, COMB, 4>(g, sino, first, i, i2, ln, wa, acc); break;
    case 5: bp_rows<ZV, CONTIG, COMB, 5>(g, sino, first, i, i2, ln, wa, acc); break;
    case 6: bp_rows<ZV, CONTIG, COMB, 6>(g, sino, first, i, i2, ln, wa, acc); break;
    default: break;
  }
}

// the rows of one angle, loaded (pk: first | count << 16; count 0: none)
template <int ZV>
struct BpRows {
  int rows;
  float t[BP_ROWS][ZV];
};
template <int ZV, bool CONTIG>
__device__ __forceinline__ void bp_load(const ParDev& g, const float* __restrict__ sino, int pk, int i,
                                        const ZLane<ZV, CONTIG>& ln, BpRows<ZV>& r) {
  r.rows = pk >> 16;
  if (r.rows == 0) return;   // wave-uniform, like the tests below
  const uint32_t row_b = 4u * (uint32_t)g.na * (uint32_t)g.nz;
  const uint32_t at = ((uint32_t)(pk & 0xffff) * (uint32_t)g.na + (uint32_t)i) * (uint32_t)g.nz;
  const __amdgpu_buffer_rsrc_t rs = buf_rsrc(sino + (size_t)at, (uint32_t)(r.rows - 1) * row_b + 4u * (uint32_t)g.nz);
#pragma unroll
  for (int k = 0; k < BP_ROWS; ++k)
    if (k < 2 || r.rows > k) zload<ZV, CONTIG>(rs, ln, k * row_b, r.t[k]);
}
template <int ZV>
__device__ __forceinline__ void bp_products(const BpRows<ZV>& r, const float2* wa, mf4 (&acc)[BP_QUADS][ZV]) {
  if (r.rows == 0) return;
#pragma unroll
  for (int k = 0; k < BP_ROWS; ++k)
    if (k < 2 || r.rows > k) {
      const float2 w = wa[k];
#pragma unroll
      for (int h = 0; h < BP_QUADS; ++h)
#pragma unroll
        for (int q = 0; q < ZV; ++q)
          acc[h][q] = __builtin_amdgcn_mfma_f32_4x4x1f32(vget(w, h), r.t[k][q], acc[h][q], 0, 0, 0);
    }
}

// lower row and weights of a pixel for one angle (np.interp; exactly at the
// last node fp[n - 1]); jr = -1: not seen
struct BpNode {
  int jr;
  float w0, w1;
};

// mirrored nodes common to both angles of a pair
__host__ __device__ __forceinline__ int bp_jlo(const ParDev& g) { return max(0, 2 * g.c + g.pair_D - (g.n - 1)); }
__host__ __device__ __forceinline__ int bp_jhi(const ParDev& g) { return min(g.n - 1, 2 * g.c + g.pair_D); }
// whether opposite angles are combined (not where the tuning's fp_pair = 0 keeps the
// plan unpaired): only where they share an interval, that is two nodes.  Of a
// single common node (n = 2, or a detector shifted by half its width) neither
// neighbour is a bin of both angles.
__host__ __device__ inline bool bp_combines(const ParDev& g) {
  return g.mu == 0.0 && g.pair_ok && g.fp_pair && bp_jhi(g) > bp_jlo(g);
}

// which nodes a pass over the angles takes: of every angle (COMB: of the pairs,
// where both angles see the pixel), or of the pixels that the pair's first or
// second angle alone sees
enum BpPass { BP_ALL = 0, BP_ONE = 1, BP_TWO = 2 };

// node of the pixel at (x, y) for angle i (COMB: unit (i, i2)) in pass PASS;
// single: only one angle of the pair sees it
template <bool COMB, int PASS>
__host__ __device__ __forceinline__ BpNode bp_node(const ParDev& g, bool on, int i, int i2, double x, double y, bool& single) {
  const BpNode none{-1, 0.f, 0.f};
  if (!on) return none;
  const int n = g.n;
  const double co = g.cs[2 * i], sn = g.cs[2 * i + 1];
  const double t = x * co - y * sn;
  int j, j1;
  float f;
  bool in = interp_node(g, t, j, j1, f);
  if constexpr (COMB) {
    if (i2 >= 0) {
      const double t2 = x * g.cs[2 * i2] - y * g.cs[2 * i2 + 1];
      int k, k1;
      float f2;
      const bool in2 = interp_node(g, t2, k, k1, f2);
      if (in != in2) {
        single = true;
        if (PASS != (in ? BP_ONE : BP_TWO)) return none;
        if (in2) {
          j = k;
          f = f2;
          in = true;
        }
      } else if (PASS != BP_ALL) {
        return none;
      } else if (in) {
        if (j < bp_jlo(g)) { j = bp_jlo(g); f = 0.0f; }
        if (j >= bp_jhi(g)) { j = bp_jhi(g) - 1; f = 1.0f; }
      }
    } else if (PASS != BP_ALL) {
      return none;
    }
  }
  if (!in) return none;
  const float aw = (!COMB && g.mu != 0.0) ? abs_weight(g, t, x * sn + y * co) : 1.0f;
  if (aw == 0.0f) return none;
  const bool last = j == n - 1;
  return BpNode{last ? j - 1 : j, last ? 0.0f : aw * (1.0f - f), last ? aw : aw * f};
}

// one pass over the angles; true: COMB, a pixel is seen by one angle of a pair
template <int ZV, bool CONTIG, bool COMB, int PASS>
__device__ __forceinline__ bool bp_pass(const ParDev& g, const float* __restrict__ sino, int r0, int c0,
                                        unsigned active, const ZLane<ZV, CONTIG>& ln, int lane,
                                        float2* tab, mf4 (&acc)[BP_QUADS][ZV]) {
  const int p = lane & 3, pa = lane >> 2;
  const double y = (double)(r0 + (p >> 1) - g.c), x = (double)(c0 + (p & 1) - g.c);
  float* const put = reinterpret_cast<float*>(tab + (pa * 4 + p) * 8);
  const float2* const get = tab + p * 8;              // this lane's pixel, angle 0
  const int steps = COMB ? g.n_units : g.na;
  bool singles = false;
#pragma unroll 1
  for (int u0 = 0; u0 < steps; u0 += 16) {
    const int u = u0 + pa;
    int i = u, i2 = -1;
    if constexpr (COMB)
      if (u < steps) {
        i = g.units[2 * u];
        i2 = g.units[2 * u + 1];
      }
    // rows of the patch's pixels at this lane's angle: their weights go to the
    // table, the first row and the row count to pk (first | rows << 16)
    BpNode nd[BP_QUADS];
    bool single = false;
    int lo = 0x7fffffff, hi = -1;
#pragma unroll
    for (int h = 0; h < BP_QUADS; ++h) {
      nd[h] = bp_node<COMB, PASS>(g, u < steps && ((active >> (4 * h + p)) & 1u), i, i2, x + (double)(2 * h), y, single);
      if (nd[h].jr >= 0) {
        lo = min(lo, nd[h].jr);
        hi = max(hi, nd[h].jr);
      }
    }
    lo = min(lo, __shfl_xor(lo, 1));
    lo = min(lo, __shfl_xor(lo, 2));
    hi = max(hi, __shfl_xor(hi, 1));
    hi = max(hi, __shfl_xor(hi, 2));
    if constexpr (COMB) singles |= __ballot(single) != 0ull;
    const int pk = hi >= 0 ? lo | ((hi + 2 - lo) << 16) : 0;
    if (PASS != BP_ALL && __ballot(pk != 0) == 0ull) continue;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < BP_QUADS; ++h) {
      const int d = nd[h].jr >= 0 ? nd[h].jr - lo : 0;
#pragma unroll
      for (int k = 0; k < BP_ROWS; ++k) put[k * BP_QUADS + h] = d == k ? nd[h].w0 : (d == k - 1 ? nd[h].w1 : 0.0f);
    }
    __builtin_amdgcn_wave_barrier();
    const int m = steps - u0 < 16 ? steps - u0 : 16;
    if constexpr (CONTIG && !COMB) {
      // the next angle's rows are loaded before this angle's products
      BpRows<ZV> even, odd;
      bp_load<ZV, CONTIG>(g, sino, rl_i(pk, 0), u0, ln, even);
#pragma unroll 1
      for (int a = 0; a < m; a += 2) {
        bp_load<ZV, CONTIG>(g, sino, a + 1 < m ? rl_i(pk, 4 * a + 4) : 0, u0 + a + 1, ln, odd);
        bp_products<ZV>(even, get + a * 32, acc);
        bp_load<ZV, CONTIG>(g, sino, a + 2 < m ? rl_i(pk, (4 * a + 8) & 63) : 0, u0 + a + 2, ln, even);
        bp_products<ZV>(odd, get + a * 32 + 32, acc);
      }
    } else {
#pragma unroll 1
      for (int a = 0; a < m; ++a) {
        const int pkv = rl_i(pk, 4 * a);
        const int ia = COMB ? rl_i(PASS == BP_TWO ? i2 : i, 4 * a) : u0 + a;
        const int ib = COMB && PASS == BP_ALL ? rl_i(i2, 4 * a) : -1;
        bp_rows_of<ZV, CONTIG, COMB && PASS == BP_ALL>(g, sino, pkv >> 16, pkv & 0xffff, ia, ib, ln, get + a * 32, acc);
      }
    }
  }
  return singles;
}

// a patch's sums
template <int ZV, bool CONTIG, bool COMB>
__device__ __forceinline__ void bp_patch(const ParDev& g, const float* __restrict__ sino, int r0, int c0,
                                         unsigned active, const ZLane<ZV, CONTIG>& ln, int lane,
                                         float2* tab, mf4 (&acc)[BP_QUADS][ZV]) {
#pragma unroll
  for (int h = 0; h < BP_QUADS; ++h)
#pragma unroll
    for (int q = 0; q < ZV; ++q) acc[h][q] = mf4{0.f, 0.f, 0.f, 0.f};
  if (active) {
    if (bp_pass<ZV, CONTIG, COMB, BP_ALL>(g, sino, r0, c0, active, ln, lane, tab, acc)) {
      bp_pass<ZV, CONTIG, true, BP_ONE>(g, sino, r0, c0, active, ln, lane, tab, acc);
      bp_pass<ZV, CONTIG, true, BP_TWO>(g, sino, r0, c0, active, ln, lane, tab, acc);
    }
  }
}

// L2-aware work order of the wavefront-uniform kernels.  About 1024 waves are
// resident per XCD at once (32 CUs x 32 waves) and consecutive logical blocks
// run on the same XCD (xcd_remap), so consecutive waves should form a compact
// tile whose data fits the XCD's 4 MB L2: forward = fp_ta consecutive angles x
// fp_tk consecutive rays (their samples at one along-ray step lie within a few
// tens of pixels), the forward's transpose = a bp_tile x bp_tile patch of 2x2
// voxel quads (detector footprint ~2.8 bp_tile bins per angle; the back
// projection's patches are listed by the plan, see bp_wave_patch).  When a ray (or
// column) spans several z chunks, the chunk is the slowest index, so that all
// resident waves share one z slab.  Padding waves exit.  Tiles never exceed
// the problem: a tile edge beyond the angle / ray / quad count would only add
// padding waves.
__host__ __device__ inline int fp_ta_eff(const ParDev& g) { return g.fp_ta < g.na ? g.fp_ta : g.na; }
__host__ __device__ inline int fp_tk_eff(const ParDev& g) { return g.fp_tk < g.n ? g.fp_tk : g.n; }
__host__ __device__ inline long long fp_tiled_rays(const ParDev& g) {
  const int ta = fp_ta_eff(g), tk = fp_tk_eff(g);
  return (long long)((g.na + ta - 1) / ta) * ((g.n + tk - 1) / tk) * ta * tk;
}
__device__ __forceinline__ bool fp_tile_ray(long long q, const ParDev& g, int& k, int& i) {
  const int ta = fp_ta_eff(g), tk = fp_tk_eff(g);
  const int ntk = (g.n + tk - 1) / tk;
  const int tsz = ta * tk;
  const long long tile = q / tsz;
  const int within = (int)(q % tsz);
  i = (int)(tile / ntk) * ta + within / tk;
  k = (int)(tile % ntk) * tk + within % tk;
  return i < g.na && k < g.n;
}
// forward's transpose: quads of 2x2 voxel columns, tiles of bp_tile x bp_tile quads
__host__ __device__ inline int bp_nquad(const ParDev& g) { return (g.n + 1) / 2; }
__host__ __device__ inline int bp_tile_eff(const ParDev& g) {
  return g.bp_tile < bp_nquad(g) ? g.bp_tile : bp_nquad(g);
}
__host__ __device__ inline long long bp_tiled_quads(const ParDev& g) {
  const int bt = bp_tile_eff(g);
  const long long t = (bp_nquad(g) + bt - 1) / bt;
  return t * t * bt * bt;
}
// upper bound of bp_tiled_quads over every tile setting (tile <= nquad)
__host__ __device__ inline long long bp_tiled_quads_max(const ParDev& g) {
  const long long e = 2ll * bp_nquad(g);
  return e * e;
}
__device__ __forceinline__ bool bp_tile_quad(long long q, const ParDev& g, int& r0, int& c0) {
  const int bt = bp_tile_eff(g);
  const int nt = (bp_nquad(g) + bt - 1) / bt;
  const int tsz = bt * bt;
  const long long tile = q / tsz;
  const int within = (int)(q % tsz);
  const int qr = (int)(tile / nt) * bt + within / bt;
  const int qc = (int)(tile % nt) * bt + within % bt;
  r0 = 2 * qr;
  c0 = 2 * qc;
  return qr < bp_nquad(g) && qc < bp_nquad(g);
}

// Back projection: the plan lists its patches of 2 rows x 4 columns (bp_list, row
// << 16 | column) along a Z curve, those with a column inside the clip circle
// first.  The wavefronts of a launch are the listed patches x z chunks, chunk
// slowest, in two groups: the active ones in equal contiguous shares per XCD
// (a compact part of the volume, whose rows its L2 holds), then the ones that
// only store zeros.  In tiles row by row without regard to the circle, the XCDs
// of the middle rows had a quarter more active patches than the mean (201 x 201 x
// 77 x 240 angles: 202 us against 154).
__host__ __device__ inline long long bp_active(const ParDev& g, int clipc) {
  return clipc ? g.bp_act : g.bp_all;
}
// blocks of BP_WAVES wavefronts: few, so that the compute units' shares differ
// by little where all wavefronts are resident at once
constexpr int BP_WAVES = 2;
__host__ __device__ inline long long bp_blocks(const ParDev& g, int clipc, int chunks, bool active) {
  const long long act = bp_active(g, clipc), w = (active ? act : g.bp_all - act) * chunks;
  return (w + BP_WAVES - 1) / BP_WAVES;
}
// wavefront w of the list -> patch and z chunk; false past its end
__device__ __forceinline__ bool bp_wave_patch(long long w, int chunks, const ParDev& g, int clipc, int& r0, int& c0,
                                              int& chunk) {
  const long long all = g.bp_all, act = bp_active(g, clipc);
  long long first = 0, count = act;
  if (w >= act * chunks) {
    if (w >= all * chunks) return false;
    w -= act * chunks;
    first = act;
    count = all - act;
  }
  chunk = (int)(w / count);
  const int at = g.bp_list[first + w % count];
  r0 = 2 * (at >> 16);
  c0 = 4 * (at & 0xffff);
  return true;
}
// the calling wavefront's place in the list; -1: none
__device__ __forceinline__ long long bp_wave(const ParDev& g, int clipc, int chunks) {
  const long long nb = bp_blocks(g, clipc, chunks, true), act = bp_active(g, clipc) * chunks;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (blockIdx.x >= nb) return act + (blockIdx.x - nb) * BP_WAVES + wv;
  const long long w = (long long)xcd_remap(blockIdx.x, (unsigned)nb) * BP_WAVES + wv;
  return w < act ? w : -1;
}
// bit 4 h + p: pixel p of quad h is inside the grid and, of those, computed
__device__ __forceinline__ void bp_patch_masks(const ParDev& g, int r0, int c0, int clipc, unsigned& inrange,
                                               unsigned& active) {
  inrange = active = 0u;
#pragma unroll
  for (int b = 0; b < 4 * BP_QUADS; ++b) {
    const int row = r0 + bp_bit_row(b), col = c0 + bp_bit_col(b);
    if (row < g.n && col < g.n) {
      inrange |= 1u << b;
      if (!(clipc && g.outside[row * g.n + col])) active |= 1u << b;
    }
  }
}
// the patch's doses: zero outside the computed columns; an infinity or a NaN (a
// row that another column of its quad skips may have held an infinity, two
// opposite rows may add past the largest number) is summed again as bp_voxel
// does it
template <int ZV, bool CONTIG>
__device__ __forceinline__ void bp_patch_store(const ParDev& g, const float* __restrict__ sino, float* vol, int r0,
                                               int c0, unsigned inrange, unsigned active,
                                               const ZLane<ZV, CONTIG>& ln, const mf4 (&acc)[BP_QUADS][ZV]) {
  bool bad = false;
#pragma unroll
  for (int h = 0; h < BP_QUADS; ++h)
#pragma unroll
    for (int q = 0; q < ZV; ++q)
#pragma unroll
      for (int p = 0; p < 4; ++p) bad |= !(fabsf(acc[h][q][p]) <= 3.4028234664e38f);
#pragma unroll
  for (int b = 0; b < 4 * BP_QUADS; ++b) {
    if (!((inrange >> b) & 1u)) continue;
    const int h = b >> 2, p = b & 3;
    float* outp = vol + ((size_t)(r0 + bp_bit_row(b)) * g.n + c0 + bp_bit_col(b)) * g.nz;
    const bool on = (active >> b) & 1u;
    if constexpr (CONTIG) {
      if (ln.z < g.nz)
        vstore<4>(outp + ln.z, on ? make_float4(acc[h][0][p], acc[h][1][p], acc[h][2][p], acc[h][3][p]) : vzero<4>());
    } else {
#pragma unroll
      for (int q = 0; q < ZV; ++q)
        if (ln.slice(q) < g.nz) outp[ln.slice(q)] = on ? acc[h][q][p] : 0.0f;
    }
  }
  if (__ballot(bad) == 0ull) return;
#pragma unroll 1
  for (int b = 0; b < 4 * BP_QUADS; ++b) {
    if (!((active >> b) & 1u)) continue;
    const int pix = (r0 + bp_bit_row(b)) * g.n + c0 + bp_bit_col(b);
#pragma unroll 1
    for (int q = 0; q < ZV; ++q) {
      const int z = ln.slice(q);
      if (z >= g.nz) continue;
      float* at = vol + (size_t)pix * g.nz + z;
      if (!(fabsf(*at) <= 3.4028234664e38f)) *at = bp_voxel<1>(g, sino, pix, z);
    }
  }
}
// how a problem's back projection lays out its slices: slices per lane (0: not
// on these kernels), 16-byte loads of four, opposite angles combined
struct BpLayout {
  int zv = 0;
  bool contig = false, comb = false;
  int chunks = 0;
};

// Global index of the calling wavefront for logical block lb.  The wave's
// slot in its block is made wave-uniform explicitly (readfirstlane), so that
// everything derived from it -- ray, angle, voxel column, geometry constants
// -- lives in scalar registers.
__device__ __forceinline__ long long wave_index(unsigned lb) {
  const int slot = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  return (long long)lb * (blockDim.x >> 6) + slot;
}

// z chunks of a wavefront: 64 lanes x ZV values; the last chunk may be
// partial (lanes past nz load from a clamped z and store nothing)
__host__ __device__ inline int wave_zchunks(int nz, int zv) { return (nz + 64 * zv - 1) / (64 * zv); }

// wave -> (ray, z chunk) of the forward kernels; false for padding waves
template <int ZV>
__device__ __forceinline__ bool fp_wave_item(long long wave, const ParDev& g, int& k, int& i, int& zc) {
  const long long rays = fp_tiled_rays(g);
  const int nch = wave_zchunks(g.nz, ZV);
  if (wave >= rays * nch) return false;
  zc = (int)(wave / rays);
  return fp_tile_ray(wave % rays, g, k, i);
}

// Paired forward work order: unit u (an angle pair, or a single angle) has
// n + pair_u extended rays e: e < n is ray e of the primary angle (with its
// partner ray when that exists), e >= n a partner-angle ray without a
// primary.  Tiles are fp_ta units x fp_tk extended rays, z chunk slowest.
__host__ __device__ inline int fp_pair_next(const ParDev& g) { return g.n + g.pair_u; }
__host__ __device__ inline int fp_pair_ta(const ParDev& g) { return g.fp_ta < g.n_units ? g.fp_ta : g.n_units; }
__host__ __device__ inline int fp_pair_tk(const ParDev& g) {
  return g.fp_tk < fp_pair_next(g) ? g.fp_tk : fp_pair_next(g);
}
__host__ __device__ inline long long fp_pair_tiled(const ParDev& g) {
  const int ta = fp_pair_ta(g), tk = fp_pair_tk(g), ne = fp_pair_next(g);
  return (long long)((g.n_units + ta - 1) / ta) * ((ne + tk - 1) / tk) * ta * tk;
}
// wave -> ray (k, i), partner ray (k2, i2) or k2 = -1, and z; ok = false for
// padding waves
struct PairItem {
  int k, i, k2, i2, zc;
  bool ok;
};
template <int ZV>
__host__ __device__ __forceinline__ PairItem fp_pair_item(long long wave, const ParDev& g) {
  PairItem it{0, 0, -1, -1, 0, false};
  const long long tiled = fp_pair_tiled(g);
  const int nch = wave_zchunks(g.nz, ZV);
  if (wave >= tiled * nch) return it;
  it.zc = (int)(wave / tiled);
  const long long q = wave % tiled;
  const int ta = fp_pair_ta(g), tk = fp_pair_tk(g), ne = fp_pair_next(g);
  const int ntk = (ne + tk - 1) / tk;
  const int tsz = ta * tk;
  const long long tile = q / tsz;
  const int within = (int)(q % tsz);
  const int u = (int)(tile / ntk) * ta + within / tk;
  const int e = (int)(tile % ntk) * tk + within % tk;
  if (u >= g.n_units || e >= ne) return it;
  const int u1 = g.units[2 * u], u2 = g.units[2 * u + 1];
  const int kk = 2 * g.c + g.pair_D - e;
  const bool has2 = e < g.n && u2 >= 0 && kk >= 0 && kk < g.n;
  if (e >= g.n && u2 < 0) return it;
  it.k = e < g.n ? e : g.pair_first2 + (e - g.n);
  it.i = e < g.n ? u1 : u2;
  it.k2 = has2 ? kk : -1;
  it.i2 = has2 ? u2 : -1;
  it.ok = true;
  return it;
}

// wave -> (voxel quad, z) of the forward's transpose; false for padding
template <int ZV>
__device__ __forceinline__ bool bp_wave_quad(long long wave, const ParDev& g, int lane, int& r0, int& c0, int& z) {
  const long long quads = bp_tiled_quads(g);
  const int nch = wave_zchunks(g.nz, ZV);
  if (wave >= quads * nch) return false;
  const int zc = (int)(wave / quads);
  if (!bp_tile_quad(wave % quads, g, r0, c0)) return false;
  z = zc * 64 * ZV + lane * ZV;
  return true;
}

// pixels of quad (r0, c0) inside the grid (bit p = pixel p) and, of those,
// the ones computed (not zeroed by the circle clip)
__device__ __forceinline__ void bp_quad_masks(const ParDev& g, int r0, int c0, int clipc, unsigned& inrange,
                                              unsigned& active) {
  inrange = 0u;
  active = 0u;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = r0 + (q >> 1), col = c0 + (q & 1);
    if (row < g.n && col < g.n) {
      inrange |= 1u << q;
      if (!(clipc && g.outside[row * g.n + col])) active |= 1u << q;
    }
  }
}

// ---------------------------------------------------------------------------
// A^T on voxel quads.  Within one angle the detector coordinates of a 2x2
// quad's voxels lie within |cos| + |sin| <= sqrt(2) of each other, so the
// candidate bins of the four voxels (fpT_voxel: floor(k*) - 1 .. + 2 each)
// span at most 6 consecutive bins.  Lane l evaluates angle i0 + l for all
// four voxels with fpT_voxel's arithmetic and writes a 6-bin x 4-voxel weight
// table to LDS; the wavefront then loads each of the angle's sinogram rows
// with a nonzero weight once for the four voxels.  Each voxel sums the same
// nonzero terms in the same order as fpT_voxel (a zero weight adds an exact
// zero), so the results are bitwise equal.
// ---------------------------------------------------------------------------
struct FpTQuadSlot {
  float4* w;   // [64][6]: bin kbase + j -> weights of the quad's voxels 0..3
  int2* kb;    // [64] first candidate bin of the angle, bit j = bin kbase + j has a nonzero weight
};
__device__ __forceinline__ FpTQuadSlot fpT_quad_slot() {
  __shared__ float4 w[4][64 * 6];
  __shared__ int2 kb[4][64];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 3;
  return {w[wv], kb[wv]};
}

template <int ZV>
__device__ __forceinline__ void fpT_quad_wave(const ParDev& g, const float* __restrict__ sino, int r0, int c0,
                                              unsigned inrange, int zl, int lane, typename VecT<ZV>::T acc[4]) {
  using V = typename VecT<ZV>::T;
  const int n = g.n;
  const size_t zstride = (size_t)g.nz;
  const FpTQuadSlot sl = fpT_quad_slot();
#pragma unroll
  for (int q = 0; q < 4; ++q) acc[q] = vzero<ZV>();
  for (int i0 = 0; i0 < g.na; i0 += 64) {
    const int i = i0 + lane;
    // the lane's own table row: cleared, then filled with the nonzero weights
    __builtin_amdgcn_wave_barrier();
    float4* const wrow = sl.w + lane * 6;
#pragma unroll
    for (int j = 0; j < 6; ++j) wrow[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    float* const wf = reinterpret_cast<float*>(wrow);
    int kbase = 0, mask = 0;
    if (i < g.na) {
      const double* M = g.mats + 6 * i;
      const double co = M[0], sn = M[1];
      int kbq[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double X = (double)(c0 + (q & 1) - g.c), Y = (double)(r0 + (q >> 1) - g.c);
        const double kstar = co * X - sn * Y + (double)g.c + g.det_offset;
        kbq[q] = (int)floor(kstar) - 1;
      }
      kbase = min(min(kbq[0], kbq[1]), min(kbq[2], kbq[3]));
#pragma unroll 1
      for (int q = 0; q < 4; ++q) {
        if (!((inrange >> q) & 1u)) continue;
        const int row = r0 + (q >> 1), col = c0 + (q & 1);
        const double X = (double)(col - g.c), Y = (double)(row - g.c);
        const double rstar = sn * X + co * Y + (double)g.c;
        const int rb = (int)floor(rstar) - 1;
        for (int d = 0; d < 4; ++d) {
          const int kk = kbq[q] + d;
          if (kk < 0 || kk >= n) continue;
          const double kp = (double)kk - g.det_offset;
          const double a0 = M[0] * kp, a1 = M[3] * kp;
          const double t = (double)(kk - g.c) - g.det_offset;
          float wk = 0.0f;
          for (int r = rb; r < rb + 4; ++r) {
            if (r < 0 || r >= n) continue;
            const double rr = (double)r;
            const double colS = (a0 + M[1] * rr) + M[2];
            const double rowS = (a1 + M[4] * rr) + M[5];
            if (!(fabs(rowS - (double)row) < 1.0 && fabs(colS - (double)col) < 1.0)) continue;
            const float wr = tap_weight_axis(rowS, row);
            const float wc = tap_weight_axis(colS, col);
            wk = __builtin_fmaf(wr * wc, abs_weight(g, t, (double)(r - g.c)), wk);
          }
          // slot kk - kbase is in 0..5: the four voxels' first bins differ by
          // <= 2 (their k* lie within |cos| + |sin| <= sqrt(2))
          const int j = kk - kbase;
          if (wk != 0.0f && j < 6) {
            wf[j * 4 + q] = wk;
            mask |= 1 << j;
          }
        }
      }
    }
    sl.kb[lane] = make_int2(kbase, mask);
    __builtin_amdgcn_wave_barrier();
    const int rows = g.na - i0 < 64 ? g.na - i0 : 64;
    for (int a = 0; a < rows; ++a) {
      const int2 km = sl.kb[a];
      const int kb0 = __builtin_amdgcn_readfirstlane(km.x);
      const int msk = __builtin_amdgcn_readfirstlane(km.y);
      const int ia = i0 + a;
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        // rows without a nonzero weight are skipped, among them every bin
        // outside 0..n-1 (its weights stay 0)
        if (!((msk >> j) & 1)) continue;
        const float4 w = sl.w[a * 6 + j];
        const V v = vload<ZV>(sino + ((size_t)(kb0 + j) * g.na + ia) * zstride + zl);
        acc[0] = vfma(w.x, v, acc[0]);
        acc[1] = vfma(w.y, v, acc[1]);
        acc[2] = vfma(w.z, v, acc[2]);
        acc[3] = vfma(w.w, v, acc[3]);
      }
    }
  }
}

// what a forward kernel does with a ray's value: store it in the sinogram, or
// the BCLP update g <- clip(g - lr * scale * value) (BCLP.py:486-487, 532)
struct StoreOut {
  float* sino;
  __device__ __forceinline__ void put(size_t at, float v) const { sino[at] = v; }
};
struct UpdateOut {
  float* gsino;
  const double* scale_p;
  float lr, glb, gub;
  __device__ __forceinline__ void put(size_t at, float v) const {
    gsino[at] = clampf(gsino[at] - lr * ((float)(*scale_p) * v), glb, gub);
  }
};

// how a problem's forward projection lays out its slices: slices per lane (0:
// not on the wavefront kernels), 64 apart or consecutive
struct FpLayout {
  int zv = 0;
  bool split = false;
};

// calls f(ZV, SPLIT, REUSE) with the layout's compile-time constants
template <class F>
void fp_dispatch(const FpLayout& l, bool reuse, F&& f) {
  using std::integral_constant;
  auto with = [&](auto r) {
    if (l.split) {
      if (l.zv == 4) f(integral_constant<int, 4>{}, std::true_type{}, r);
      else if (l.zv == 3) f(integral_constant<int, 3>{}, std::true_type{}, r);
      else f(integral_constant<int, 2>{}, std::true_type{}, r);
    } else {
      if (l.zv == 4) f(integral_constant<int, 4>{}, std::false_type{}, r);
      else if (l.zv == 2) f(integral_constant<int, 2>{}, std::false_type{}, r);
      else f(integral_constant<int, 1>{}, std::false_type{}, r);
    }
  };
  if (reuse) with(std::true_type{});
  else with(std::false_type{});
}

// calls f(ZV, CONTIG, COMB) with the layout's compile-time constants
template <class F>
void bp_dispatch(const BpLayout& l, F&& f) {
  using std::integral_constant;
  auto with = [&](auto comb) {
    if (l.contig) f(integral_constant<int, 4>{}, std::true_type{}, comb);
    else if (l.zv == 4) f(integral_constant<int, 4>{}, std::false_type{}, comb);
    else if (l.zv == 3) f(integral_constant<int, 3>{}, std::false_type{}, comb);
    else if (l.zv == 2) f(integral_constant<int, 2>{}, std::false_type{}, comb);
    else f(integral_constant<int, 1>{}, std::false_type{}, comb);
  };
  if (l.comb) with(std::true_type{});
  else with(std::false_type{});
}

// host helpers implemented in parallel.hip
int par_slice_minmax(vamx_plan* p, const float* vol, hipStream_t s);
int par_forward_launch(vamx_plan* p, const float* vol, float* sino, hipStream_t s, bool warp_clip);
int par_backward_launch(vamx_plan* p, const float* sino, float* vol, hipStream_t s, bool clipc);
BpLayout bp_layout(const vamx_plan* p, uintptr_t align_bits, int problems = 1);   // problems: of one launch
bool par_use_vec4(const vamx_plan* p, const void* a, const void* b);
bool par_use_vec2(const vamx_plan* p, const void* a, const void* b);
int par_wave_zv(const vamx_plan* p, const void* a, const void* b, int requested);
FpLayout fp_layout(const vamx_plan* p, uintptr_t align_bits);
int wave_zv_choice(int nz, uintptr_t align_bits, int requested);
void par_pair_units(const std::vector<double>& cs, int na, int n, int c, double D, std::vector<int>& units,
                    int& npaired_rays, int& first2);
// Problems of a batch that share one launch of a forward, thin or inclined kernel:
// those of one class (kernel, lanes, slices per lane, wavefronts per block).  A block finds
// its problem by its number; the table is on the device, the buffers come with the
// launch.
constexpr int kBatchChunk = 64;   // problems per launch
struct InclShift {
  int lo = 0, rows = 0;   // least shift of a ray's samples, detector rows of a wavefront
};
struct LaneProblem {
  ParDev g;
  const float* minmax;
  int clip, pair;
  InclShift shift;
};
struct LaneTable {
  const LaneProblem* items;
  int m;
  unsigned begin[kBatchChunk];   // first block of each
  const float* in[kBatchChunk];
  float* out[kBatchChunk];
};
// the calling block's problem and its number there; each XCD takes a contiguous
// share of the problems' blocks
__device__ __forceinline__ int lane_problem(const LaneTable& t, unsigned& lb) {
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  int lo = 0, hi = t.m - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (t.begin[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  lb = b - t.begin[lo];
  return lo;
}
struct LaneClass {
  int key = 0;                // 0: none
  long long blocks = 0, waves = 0;
  LaneProblem problem{};
};
// inclined projections on wavefronts (incl.hip)
bool incl_wave_ok(const vamx_plan* p);
int incl_forward_store(vamx_plan* p, const float* vol, float* sino, hipStream_t s);
int incl_forward_update(vamx_plan* p, const float* vol, const UpdateOut& out, hipStream_t s);
int incl_backward(vamx_plan* p, const float* sino, float* vol, bool clipc, hipStream_t s);
LaneClass incl_class(const vamx_plan* p, bool forward, bool clip);
int incl_batch(int key, const LaneTable& t, unsigned blocks, hipStream_t s);
// thin problems at zero inclination (thin.hip); the forward reads the plan's
// slice min / max when clip is set
bool thin_ok(const vamx_plan* p);
int thin_forward_store(vamx_plan* p, const float* vol, float* sino, bool clip, hipStream_t s);
int thin_forward_update(vamx_plan* p, const float* vol, const UpdateOut& out, bool clip, hipStream_t s);
int thin_backward(vamx_plan* p, const float* sino, float* vol, bool clipc, hipStream_t s);
LaneClass thin_class(const vamx_plan* p, const void* in, const void* out, bool forward, bool clip);
int thin_batch(int key, const LaneTable& t, unsigned blocks, hipStream_t s);

}  // namespace vamx
