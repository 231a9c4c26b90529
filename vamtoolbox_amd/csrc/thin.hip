// Thin problems (few slices, down to one) at zero inclination on wavefronts.
//
// With fewer than 32 slices one ray (voxel column) leaves most lanes of a
// wavefront idle, so the lanes form G = 64 / L groups of L, and a lane holds
// ZV slices (L ZV >= nz).
//   forward: a wavefront owns a ray -- and its opposite ray, from the same
//     taps -- and group g takes every G-th sample; the groups' sums are added
//     at the end.  Lane l evaluates sample r0 + l's float64 geometry once for
//     all slices, into a per-wavefront LDS table (one slice: a lane uses its
//     own sample directly).
//   back: group g owns a voxel column of an 8 x 8 patch; its lanes evaluate L
//     angles at a time into the table.  Where the columns alone would leave
//     the GPU short of wavefronts, the wavefronts of a block split the angles
//     and add their sums through LDS.
// The per-lane kernels evaluate every sample's geometry in every lane and
// walk a whole ray (all angles) serially per thread, which leaves a small
// problem waiting on one chain of loads per thread.
#include <type_traits>

#include "par_core.h"

namespace vamx {

namespace {

// table entries per step: eight tap loads in flight, and registers for 6 or
// more wavefronts per SIMD (four steps of 16-byte taps held 152 registers)
template <int ZV> constexpr int steps() { return ZV == 4 ? 2 : 4; }
constexpr int kTab = 64 + 4 * 32;      // entries past 64 are empty
constexpr int kOne = 1 << 28;          // cell flags: one column (kOne) or row (2 kOne) only
constexpr uint32_t kOut = 0x80000000u; // offset past every buffer: the load returns 0

// the taps of one axis: first one b with weight s0, and b + 1 with s1 (0: no
// second tap -- it is not read, its voxels may lie outside or hold no number)
__device__ __forceinline__ void axis_taps(double coord, int n, int& b, double& s0, double& s1) {
  const double f = floor(coord), d = coord - f;
  const int fi = (int)f;
  b = fi < 0 ? 0 : fi;
  s0 = fi < 0 ? d : 1.0 - d;
  s1 = fi < 0 || fi >= n - 1 ? 0.0 : d;
}

// abs_weight (par_core.h) with the half chord of a ray taken once
struct Chord {
  bool in;
  double half;
};
__device__ __forceinline__ Chord chord_of(const ParDev& g, double t) {
  if (g.mu == 0.0) return {true, 0.0};
  return {fabs(t) < g.radius, sqrt(fmax(0.0, g.radius * g.radius - t * t))};
}
__device__ __forceinline__ float chord_weight(const ParDev& g, const Chord& c, double s) {
  if (g.mu == 0.0) return 1.0f;
  return c.in ? expf((float)(-g.mu * (fmax(0.0, c.half - s) * g.inv_cos))) : 0.0f;
}

// one sample of a ray: cell (with its flags), the axes' weights, the rays' absorption
struct Sample {
  int base;
  float r0, r1, c0, c1, a, a2;
  bool valid;
};
template <bool PAIR>
__device__ __forceinline__ Sample ray_sample(const ParDev& g, const double* M, double a0, double a1, const Chord& ch,
                                             int r, int r2_lo) {
  Sample s{0, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, false};
  const int n = g.n;
  const double rr = (double)r;
  const double col = (a0 + M[1] * rr) + M[2];
  const double row = (a1 + M[4] * rr) + M[5];
  if (!(row > -1.0 && row < (double)n && col > -1.0 && col < (double)n)) return s;
  int br, bc;
  double r0w, r1w, c0w, c1w;
  axis_taps(row, n, br, r0w, r1w);
  axis_taps(col, n, bc, c0w, c1w);
  if (!PAIR || r < n) s.a = chord_weight(g, ch, (double)(r - g.c));
  if constexpr (PAIR)
    if (r >= r2_lo) s.a2 = chord_weight(g, ch, (double)(g.c - r));
  s.valid = s.a != 0.0f || s.a2 != 0.0f;
  s.base = (br * n + bc) | (c1w == 0.0 ? kOne : 0) | (r1w == 0.0 ? 2 * kOne : 0);
  s.r0 = (float)r0w;
  s.r1 = (float)r1w;
  s.c0 = (float)c0w;
  s.c1 = (float)c1w;
  return s;
}

struct FpThinSlot {
  float4* w;   // the axes' weights r0 r1 c0 c1
  float4* a;   // absorption (ray, partner ray), cell, whether it is a sample
};
__device__ __forceinline__ FpThinSlot fp_thin_slot() {
  __shared__ float4 w[4][kTab];
  __shared__ float4 a[4][kTab];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 3;
  return {w[wv], a[wv]};
}

// a sample from its taps, clipped to the slice range
template <int ZV, bool CLIP>
__device__ __forceinline__ typename VecT<ZV>::T thin_value(const typename VecT<ZV>::T (&t)[4], float r0, float r1,
                                                           float c0, float c1, const typename VecT<ZV>::T& lo,
                                                           const typename VecT<ZV>::T& hi) {
  using V = typename VecT<ZV>::T;
  V v = vfma(r1 * c1, t[3], vfma(r1 * c0, t[2], vfma(r0 * c1, t[1], vmul(r0 * c0, t[0]))));
  if constexpr (CLIP) v = vclamp(v, lo, hi);
  return v;
}

// its taps at byte offset zb into the columns; a buffer descriptor over the
// whole volume keeps the addresses to 32-bit offsets (thin_ok)
template <int ZV>
__device__ __forceinline__ void thin_load(__amdgpu_buffer_rsrc_t vol, int base, uint32_t row_b, uint32_t col_b,
                                          uint32_t zb, typename VecT<ZV>::T (&t)[4]) {
  const uint32_t p = (uint32_t)(base & (kOne - 1)) * col_b + zb;
  const uint32_t o1 = base & kOne ? kOut : p + col_b, o2 = base & (2 * kOne) ? kOut : p + row_b;
  const uint32_t o3 = base & (3 * kOne) ? kOut : p + row_b + col_b;
  t[0] = bload<ZV>(vol, p, 0);
  t[1] = bload<ZV>(vol, o1, 0);
  t[2] = bload<ZV>(vol, o2, 0);
  t[3] = bload<ZV>(vol, o3, 0);
}

// R > 1 (L = 1): the wavefront's lanes are R neighbouring rays (k, per lane)
// x 64 / R samples
template <int ZV, int L, int R, bool CLIP, bool PAIR>
__device__ __forceinline__ void thin_ray(const ParDev& g, const float* __restrict__ vol,
                                         const float* __restrict__ minmax, int k, int i, int z, int lane,
                                         typename VecT<ZV>::T& acc, typename VecT<ZV>::T& acc2) {
  using V = typename VecT<ZV>::T;
  static_assert(!(PAIR && CLIP), "the clipped sample is discontinuous at the border: no pairing");
  constexpr int G = 64 / L, kU = steps<ZV>();
  const int n = g.n, nz = g.nz, grp = lane / L;
  const __amdgpu_buffer_rsrc_t vr = buf_rsrc(vol, (uint32_t)n * (uint32_t)n * (uint32_t)nz * 4u);
  const uint32_t col_b = 4u * (uint32_t)nz, row_b = (uint32_t)n * col_b, zb = 4u * (uint32_t)z;
  const double* M = g.mats + 6 * i;
  const double kp = (double)k - g.det_offset;
  const double a0 = M[0] * kp, a1 = M[3] * kp;
  const Chord ch = chord_of(g, (double)(k - g.c) - g.det_offset);
  V lo = vzero<ZV>(), hi = vzero<ZV>();
  if constexpr (CLIP) {
    lo = vload<ZV>(minmax + z);
    hi = vload<ZV>(minmax + nz + z);
  }
  acc = vzero<ZV>();
  acc2 = vzero<ZV>();
  // samples of the ray and of its opposite ray (fp_ray_wave)
  const int r_end = PAIR ? (2 * g.c + 1 > n ? 2 * g.c + 1 : n) : n;
  const int r2_lo = 2 * g.c - n + 1;
  if constexpr (L == 1) {
    for (int r = lane / R; r < r_end; r += 64 / R) {
      const Sample s = ray_sample<PAIR>(g, M, a0, a1, ch, r, r2_lo);
      if (!s.valid) continue;
      V t[4];
      thin_load<ZV>(vr, s.base, row_b, col_b, zb, t);
      const V v = thin_value<ZV, CLIP>(t, s.r0, s.r1, s.c0, s.c1, lo, hi);
      acc = vfma(s.a, v, acc);
      if constexpr (PAIR) acc2 = vfma(s.a2, v, acc2);
    }
  } else {
    const FpThinSlot sl = fp_thin_slot();
    for (int p = lane; p < kTab - 64; p += 64) sl.a[64 + p] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int r0 = 0; r0 < r_end; r0 += 64) {
      Sample s{0, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, false};
      if (r0 + lane < r_end) s = ray_sample<PAIR>(g, M, a0, a1, ch, r0 + lane, r2_lo);
      const unsigned long long m = __ballot(s.valid);
      __builtin_amdgcn_wave_barrier();
      sl.w[lane] = make_float4(s.r0, s.r1, s.c0, s.c1);
      sl.a[lane] = make_float4(s.a, s.a2, __int_as_float(s.base), s.valid ? 1.0f : 0.0f);
      __builtin_amdgcn_wave_barrier();
      if (!m) continue;
      const int first = __builtin_ctzll(m) & ~(G - 1), last = 63 - __builtin_clzll(m);
      for (int e0 = first; e0 <= last; e0 += kU * G) {
        V t[kU][4];
        float4 w[kU], a[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int e = e0 + u * G + grp;
          a[u] = sl.a[e];
          w[u] = sl.w[e];
          if (a[u].w != 0.0f) thin_load<ZV>(vr, __float_as_int(a[u].z), row_b, col_b, zb, t[u]);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          if (a[u].w == 0.0f) continue;
          const V v = thin_value<ZV, CLIP>(t[u], w[u].x, w[u].y, w[u].z, w[u].w, lo, hi);
          acc = vfma(a[u].x, v, acc);
          if constexpr (PAIR) acc2 = vfma(a[u].y, v, acc2);
        }
      }
    }
  }
#pragma unroll
  for (int o = L * R; o < 64; o <<= 1) {
#pragma unroll
    for (int q = 0; q < ZV; ++q) {
      vset(acc, q, vget(acc, q) + __shfl_xor(vget(acc, q), o));
      if constexpr (PAIR) vset(acc2, q, vget(acc2, q) + __shfl_xor(vget(acc2, q), o));
    }
  }
}

template <int ZV>
__device__ __forceinline__ bool thin_finite(const typename VecT<ZV>::T& v) {
  bool ok = true;
#pragma unroll
  for (int q = 0; q < ZV; ++q) ok &= fabsf(vget(v, q)) <= 3.4028234664e38f;
  return ok;
}
// A ray and its opposite ray (k2 < 0: none) from the same taps.  The two samples at
// the ends of a pair that belong to one of the rays count for the other with weight
// 0, which a voxel without a finite value turns into a NaN: where a sum is not
// finite, the rays are walked one by one (all lanes take part) and replace such sums.
template <int ZV, int L, int R>
__device__ __forceinline__ void thin_pair_rays(const ParDev& g, const float* __restrict__ vol,
                                               const float* __restrict__ minmax, int k, int i, int k2, int i2, int z,
                                               int lane, typename VecT<ZV>::T& acc, typename VecT<ZV>::T& acc2) {
  using V = typename VecT<ZV>::T;
  thin_ray<ZV, L, R, false, true>(g, vol, minmax, k, i, z, lane, acc, acc2);
  if (__ballot(!thin_finite<ZV>(acc) || !thin_finite<ZV>(acc2)) == 0ull) return;
#pragma unroll 1
  for (int h = 0; h < 2; ++h) {
    V alone, none;
    thin_ray<ZV, L, R, false, false>(g, vol, minmax, h && k2 >= 0 ? k2 : k, h && k2 >= 0 ? i2 : i, z, lane, alone, none);
    V& sum = h ? acc2 : acc;
#pragma unroll
    for (int q = 0; q < ZV; ++q)
      if (!(fabsf(vget(sum, q)) <= 3.4028234664e38f)) vset(sum, q, vget(alone, q));
  }
}

// one block's rays, lb the block's number in the problem
template <int ZV, int L, int R, class Out>
__device__ __forceinline__ void thin_fp_block(const ParDev& g, const float* __restrict__ vol,
                                              const float* __restrict__ minmax, int clip, int pair, const Out& out,
                                              unsigned lb) {
  using V = typename VecT<ZV>::T;
  static_assert(R == 1 || L == 1, "several rays per wavefront: one lane per ray and sample");
  const int lane = threadIdx.x & 63, z = (lane & (L - 1)) * ZV;
  const int zl = z < g.nz ? z : g.nz - ZV;   // lanes past nz read a copy and store nothing
  const long long wave = wave_index(lb);
  int k, i, k2 = -1, i2 = -1;
  if constexpr (R > 1) {
    // wavefronts in ray order; a lane without a ray of its own walks the last
    // one again and stores nothing.  e, k2: extended rays as in fp_pair_item
    const int ne = pair ? fp_pair_next(g) : g.n, nu = pair ? g.n_units : g.na, nw = (ne + R - 1) / R;
    if (wave >= (long long)nw * nu) return;   // whole wavefronts
    const int u = (int)(wave / nw), e = (int)(wave % nw) * R + lane % R;
    int store = e < ne ? 1 : 0;
    const int ee = e < ne ? e : ne - 1;
    k = ee;
    i = u;
    if (pair) {
      const int u1 = g.units[2 * u], u2 = g.units[2 * u + 1], kk = 2 * g.c + g.pair_D - ee;
      const bool extra = ee >= g.n;            // a partner-angle ray without a primary
      if (extra && u2 < 0) store = 0;
      k = extra ? g.pair_first2 + (ee - g.n) : ee;
      i = extra && u2 >= 0 ? u2 : u1;
      if (extra && u2 < 0) k = g.n - 1;
      k2 = !extra && u2 >= 0 && kk >= 0 && kk < g.n ? kk : -1;
      i2 = u2;
    }
    const bool clip_on = clip && wave_clip_active<ZV>(vload<ZV>(minmax + zl), vload<ZV>(minmax + g.nz + zl));
    const bool first = lane < R && store;
    V acc, acc2;
    if (clip_on) {
      thin_ray<ZV, L, R, true, false>(g, vol, minmax, k, i, zl, lane, acc, acc2);
      if (first) out.put(((size_t)k * g.na + i) * g.nz, vget(acc, 0));
      if (__ballot(k2 >= 0)) {
        const int kh = k2 >= 0 ? k2 : k, ih = k2 >= 0 ? i2 : i;
        thin_ray<ZV, L, R, true, false>(g, vol, minmax, kh, ih, zl, lane, acc, acc2);
        if (first && k2 >= 0) out.put(((size_t)k2 * g.na + i2) * g.nz, vget(acc, 0));
      }
    } else {
      thin_pair_rays<ZV, L, R>(g, vol, minmax, k, i, k2, i2, zl, lane, acc, acc2);
      if (first) out.put(((size_t)k * g.na + i) * g.nz, vget(acc, 0));
      if (first && k2 >= 0) out.put(((size_t)k2 * g.na + i2) * g.nz, vget(acc2, 0));
    }
    return;
  }
  if (pair) {
    const PairItem it = fp_pair_item<1>(wave, g);
    if (!it.ok) return;
    k = it.k;
    i = it.i;
    k2 = it.k2;
    i2 = it.i2;
  } else {
    if (wave >= fp_tiled_rays(g) || !fp_tile_ray(wave, g, k, i)) return;   // whole wavefronts
  }
  const bool clip_on = clip && wave_clip_active<ZV>(vload<ZV>(minmax + zl), vload<ZV>(minmax + g.nz + zl));
  auto put = [&](int kh, int ih, const V& v) {
    if (lane < L && z < g.nz) {
#pragma unroll
      for (int q = 0; q < ZV; ++q) out.put(((size_t)kh * g.na + ih) * g.nz + z + q, vget(v, q));
    }
  };
  V acc, acc2;
  if (clip_on) {
    for (int h = 0; h < (k2 >= 0 ? 2 : 1); ++h) {
      const int kh = h ? k2 : k, ih = h ? i2 : i;
      thin_ray<ZV, L, 1, true, false>(g, vol, minmax, kh, ih, zl, lane, acc, acc2);
      put(kh, ih, acc);
    }
  } else if (k2 >= 0) {
    thin_pair_rays<ZV, L, 1>(g, vol, minmax, k, i, k2, i2, zl, lane, acc, acc2);
    put(k, i, acc);
    put(k2, i2, acc2);
  } else {
    thin_ray<ZV, L, 1, false, false>(g, vol, minmax, k, i, zl, lane, acc, acc2);
    put(k, i, acc);
  }
}

template <int ZV, int L, int R, class Out>
__global__ __launch_bounds__(256) void thin_fp_kernel(ParDev g, const float* __restrict__ vol,
                                                      const float* __restrict__ minmax, int clip, int pair, Out out) {
  thin_fp_block<ZV, L, R>(g, vol, minmax, clip, pair, out, xcd_remap(blockIdx.x, gridDim.x));
}
template <int ZV, int L>
__global__ __launch_bounds__(256) void thin_fp_batch_kernel(LaneTable t) {
  unsigned lb;
  const int p = lane_problem(t, lb);
  const LaneProblem& q = t.items[p];
  thin_fp_block<ZV, L, 1>(q.g, t.in[p], q.minmax, q.clip, q.pair, StoreOut{t.out[p]}, lb);
}

// one block's columns, lb the block's number in the problem
template <int ZV, int L>
__device__ __forceinline__ void thin_bp_block(const ParDev& g, const float* __restrict__ sino, float* __restrict__ vol,
                                              int clipc, unsigned lb) {
  using V = typename VecT<ZV>::T;
  constexpr int G = 64 / L, kAng = 4;
  // per wavefront: its table of 64 entries (L > 1) and its lanes' sums
  extern __shared__ float4 thin_bp_lds[];
  const int lane = threadIdx.x & 63, l = lane & (L - 1), grp = lane / L;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), split = blockDim.x >> 6;
  const int n = g.n, nz = g.nz, nt = (n + 7) / 8;
  const int z = l * ZV, zl = z < nz ? z : nz - ZV;
  // block -> G columns of an 8 x 8 patch
  const int patch = (int)(lb / (64 / G)), in = (int)(lb % (64 / G)) * G + grp;
  const int row = (patch / nt) * 8 + (in >> 3), col = (patch % nt) * 8 + (in & 7);
  const bool inside = row < n && col < n;
  const bool active = inside && !(clipc && g.outside[row * n + col]);
  const double x = (double)(col - g.c), y = (double)(row - g.c);
  const int i_end = (int)((long long)g.na * (wv + 1) / split);
  V acc = vzero<ZV>();
  const __amdgpu_buffer_rsrc_t sr = buf_rsrc(sino, (uint32_t)n * (uint32_t)g.na * (uint32_t)nz * 4u);
  const uint32_t bin_b = 4u * (uint32_t)nz, row_b = (uint32_t)g.na * bin_b;
  // row weights and the byte offsets of the two rows of angle i (np.interp as
  // in interp_node; the fraction is taken from the distance to the first
  // node): kOut where a row is not read -- no ray, a column that is not
  // computed, no absorption weight, past the last node
  auto geom = [&](int i, float& w0, float& w1, uint32_t& p0, uint32_t& p1) {
    w0 = w1 = 0.0f;
    p0 = p1 = kOut;
    const int ic = i < i_end ? i : i_end - 1;
    const double co = g.cs[2 * ic], sn = g.cs[2 * ic + 1];
    const double t = x * co - y * sn;
    if (!active || i >= i_end || !(t >= g.xp0 && t <= g.xp_last)) return;
    const double u = t - g.xp0, fl = floor(u);
    const int j = min((int)fl, n - 1);
    const float w = (float)(u - fl);
    float aw = 1.0f;
    if (g.mu != 0.0) {
      aw = abs_weight(g, t, x * sn + y * co);
      if (aw == 0.0f) return;
    }
    w0 = aw * (1.0f - w);
    w1 = aw * w;
    p0 = ((uint32_t)j * (uint32_t)g.na + (uint32_t)i) * bin_b;
    p1 = j < n - 1 ? p0 + row_b : kOut;
  };
  // the angles of a step are summed from zero and added once: the sum so far,
  // whose rounding is what the error is made of, is rounded once a step, not
  // twice an angle
  int i = (int)((long long)g.na * wv / split);
  if constexpr (L == 1) {
    const uint32_t zb = 4u * (uint32_t)zl;
    for (; i < i_end; i += kAng) {
      V b0[kAng], b1[kAng];
      float w0[kAng], w1[kAng];
#pragma unroll
      for (int u = 0; u < kAng; ++u) {
        uint32_t p0, p1;
        geom(i + u, w0[u], w1[u], p0, p1);
        b0[u] = bload<ZV>(sr, p0 + zb, 0);
        b1[u] = bload<ZV>(sr, p1 + zb, 0);
      }
      V part = vfma(w1[0], b1[0], vmul(w0[0], b0[0]));
#pragma unroll
      for (int u = 1; u < kAng; ++u) part = vfma(w1[u], b1[u], vfma(w0[u], b0[u], part));
      acc = vadd(acc, part);
    }
  } else {
    float4* const tb = thin_bp_lds + wv * 64;
    const uint32_t zb = 4u * (uint32_t)zl;
    for (; i < i_end; i += L) {
      float w0, w1;
      uint32_t p0, p1;
      geom(i + l, w0, w1, p0, p1);
      __builtin_amdgcn_wave_barrier();
      tb[lane] = make_float4(w0, w1, __uint_as_float(p0), __uint_as_float(p1));
      __builtin_amdgcn_wave_barrier();
      constexpr int K = L < kAng ? L : kAng;
#pragma unroll
      for (int u0 = 0; u0 < L; u0 += K) {
        if (u0 > 0 && i + u0 >= i_end) break;
        V b0[K], b1[K];
        float4 e[K];
#pragma unroll
        for (int u = 0; u < K; ++u) {
          e[u] = tb[grp * L + u0 + u];
          b0[u] = bload<ZV>(sr, __float_as_uint(e[u].z) + zb, 0);
          b1[u] = bload<ZV>(sr, __float_as_uint(e[u].w) + zb, 0);
        }
        V part = vfma(e[0].y, b1[0], vmul(e[0].x, b0[0]));
#pragma unroll
        for (int u = 1; u < K; ++u) part = vfma(e[u].y, b1[u], vfma(e[u].x, b0[u], part));
        acc = vadd(acc, part);
      }
    }
  }
  if (split > 1) {
    float* const sums = reinterpret_cast<float*>(thin_bp_lds + (L == 1 ? 0 : blockDim.x));
#pragma unroll
    for (int q = 0; q < ZV; ++q) sums[q * blockDim.x + threadIdx.x] = vget(acc, q);
    __syncthreads();
    if (wv == 0) {
      for (int s = 1; s < split; ++s)
#pragma unroll
        for (int q = 0; q < ZV; ++q) vset(acc, q, vget(acc, q) + sums[q * blockDim.x + s * 64 + lane]);
    }
  }
  if (wv == 0 && inside && z < nz) vstore<ZV>(vol + ((size_t)row * n + col) * nz + z, acc);
}

template <int ZV, int L>
__global__ __launch_bounds__(1024) void thin_bp_kernel(ParDev g, const float* __restrict__ sino,
                                                       float* __restrict__ vol, int clipc) {
  thin_bp_block<ZV, L>(g, sino, vol, clipc, xcd_remap(blockIdx.x, gridDim.x));
}
template <int ZV, int L>
__global__ __launch_bounds__(1024) void thin_bp_batch_kernel(LaneTable t) {
  unsigned lb;
  const int p = lane_problem(t, lb);
  const LaneProblem& q = t.items[p];
  thin_bp_block<ZV, L>(q.g, t.in[p], t.out[p], q.clip, lb);
}

// z layout: four slices per lane where nz is a multiple of 4 and the buffers are
// 16-byte aligned, else one.  Forward and back with four, and with one: 200 x 200 x
// 24, 180 angles 86 + 59 and 106 + 67 us, x 4 32 + 23 and 42 + 25, 512 x 512 x 4, 360
// angles 277 + 240 and 360 + 277; 200 x 200 x 8 49 + 35 and 48 + 33.
bool thin_v4(int nz, const void* a, const void* b) {
  return nz % 4 == 0 && ((uintptr_t)a | (uintptr_t)b) % 16 == 0;
}

// lanes that hold a problem's slices
int thin_lanes(int nz, bool v4) {
  const int lanes = v4 ? nz / 4 : nz;
  int l = 1;
  while (l < lanes) l *= 2;
  return l;
}

template <class F>
void thin_dispatch(int lanes, bool v4, F&& f) {
  using std::integral_constant;
  auto with = [&](auto zv) {
    if (lanes == 1) f(zv, integral_constant<int, 1>{});
    else if (lanes == 2) f(zv, integral_constant<int, 2>{});
    else if (lanes == 4) f(zv, integral_constant<int, 4>{});
    else if (lanes == 8) f(zv, integral_constant<int, 8>{});
    else if (lanes == 16) f(zv, integral_constant<int, 16>{});
    else f(zv, integral_constant<int, 32>{});
  };
  if (v4) with(integral_constant<int, 4>{});
  else with(integral_constant<int, 1>{});
}

// opposite rays share their taps' loads, but below about 4 wavefronts per SIMD the
// GPU has room to project them side by side instead
int thin_pair(const ParDev& g) { return g.fp_pair && g.pair_ok && fp_pair_tiled(g) >= 4096; }

// one slice: 8 neighbouring rays x 8 samples per wavefront, whose taps lie in a
// patch of about 11 x 11 voxels (64 samples of one ray can touch 64 cache lines),
// where that still leaves 4 wavefronts per SIMD; 0: not so
long long thin_waves8(const ParDev& g) {
  const int pair = thin_pair(g), nu = pair ? g.n_units : g.na, ne = pair ? fp_pair_next(g) : g.n;
  const long long waves = (long long)nu * ((ne + 7) / 8);
  return g.nz == 1 && waves >= 4096 ? waves : 0;
}

// back projection: blocks, and wavefronts per block -- the angles are split until
// about 8 wavefronts per SIMD are in flight, at most 16 ways and into no fewer than
// 8 angles
long long thin_bp_blocks(const ParDev& g, int lanes) { return ((g.n + 7) / 8) * (long long)((g.n + 7) / 8) * lanes; }
int thin_bp_split(const ParDev& g, long long blocks) {
  int split = 1;
  while (split < 16 && blocks * split < 8192 && g.na >= 16 * split) split *= 2;
  return split;
}
template <int ZV, int L>
size_t thin_bp_lds_bytes(int split) {
  return (L == 1 ? 0 : 64 * split * sizeof(float4)) + (split > 1 ? 64 * split * ZV * sizeof(float) : 0);
}

template <class Out>
int thin_forward(vamx_plan* p, const float* vol, const void* sino, Out out, bool clip, hipStream_t s) {
  const ParDev& g = p->par;
  const int pair = thin_pair(g);
  if (const long long waves8 = thin_waves8(g)) {
    hipLaunchKernelGGL((thin_fp_kernel<1, 1, 8, Out>), dim3(blocks_for(waves8 * 64, 256)), dim3(256), 0, s, g, vol,
                       p->d_minmax, clip ? 1 : 0, pair, out);
    VAMX_HIP(hipGetLastError());
    return VAMX_OK;
  }
  const long long waves = pair ? fp_pair_tiled(g) : fp_tiled_rays(g);
  const bool v4 = thin_v4(g.nz, vol, sino);
  thin_dispatch(thin_lanes(g.nz, v4), v4, [&](auto zv, auto l) {
    constexpr int ZV = decltype(zv)::value, L = decltype(l)::value;
    hipLaunchKernelGGL((thin_fp_kernel<ZV, L, 1, Out>), dim3(blocks_for(waves * 64, 256)), dim3(256), 0, s, g, vol,
                       p->d_minmax, clip ? 1 : 0, pair, out);
  });
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

}  // namespace

bool thin_ok(const vamx_plan* p) {
  const ParDev& g = p->par;
  // 32-bit byte offsets into the volume and the sinogram
  const double most = 4.0 * g.n * (double)(g.n > g.na ? g.n : g.na) * g.nz;
  return !g.incl && !g.occ && g.n >= 2 && g.nz < 32 && most < 2147483648.0 && !(p->flags & VAMX_PAR_PER_LANE_GEOMETRY);
}

int thin_forward_store(vamx_plan* p, const float* vol, float* sino, bool clip, hipStream_t s) {
  return thin_forward(p, vol, sino, StoreOut{sino}, clip, s);
}

int thin_forward_update(vamx_plan* p, const float* vol, const UpdateOut& out, bool clip, hipStream_t s) {
  return thin_forward(p, vol, out.gsino, out, clip, s);
}

int thin_backward(vamx_plan* p, const float* sino, float* vol, bool clipc, hipStream_t s) {
  const ParDev& g = p->par;
  const bool v4 = thin_v4(g.nz, sino, vol);
  thin_dispatch(thin_lanes(g.nz, v4), v4, [&](auto zv, auto l) {
    constexpr int ZV = decltype(zv)::value, L = decltype(l)::value;
    const long long blocks = thin_bp_blocks(g, L);
    const int split = thin_bp_split(g, blocks);
    hipLaunchKernelGGL((thin_bp_kernel<ZV, L>), dim3((unsigned)blocks), dim3(64 * split),
                       (thin_bp_lds_bytes<ZV, L>(split)), s, g, sino, vol, clipc ? 1 : 0);
  });
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

// class of a problem: 1 << 16, 1 << 15 forward, 1 << 14 four slices per lane,
// wavefronts per block << 8, lanes
LaneClass thin_class(const vamx_plan* p, const void* in, const void* out, bool forward, bool clip) {
  const ParDev& g = p->par;
  LaneClass c;
  if (!thin_ok(p) || (forward && thin_waves8(g))) return c;
  const bool v4 = thin_v4(g.nz, in, out);
  const int lanes = thin_lanes(g.nz, v4);
  c.problem.g = g;
  c.problem.minmax = p->d_minmax;
  c.problem.clip = clip;
  int per_block = 4;
  if (forward) {
    c.problem.pair = thin_pair(g);
    c.waves = c.problem.pair ? fp_pair_tiled(g) : fp_tiled_rays(g);
    c.blocks = (c.waves + 3) / 4;
  } else {
    c.blocks = thin_bp_blocks(g, lanes);
    per_block = thin_bp_split(g, c.blocks);
    c.waves = c.blocks * per_block;
  }
  c.key = 1 << 16 | (forward ? 1 << 15 : 0) | (v4 ? 1 << 14 : 0) | per_block << 8 | lanes;
  return c;
}

int thin_batch(int key, const LaneTable& t, unsigned blocks, hipStream_t s) {
  const int per_block = key >> 8 & 31;
  thin_dispatch(key & 63, key >> 14 & 1, [&](auto zv, auto l) {
    constexpr int ZV = decltype(zv)::value, L = decltype(l)::value;
    if (key >> 15 & 1)
      hipLaunchKernelGGL((thin_fp_batch_kernel<ZV, L>), dim3(blocks), dim3(256), 0, s, t);
    else
      hipLaunchKernelGGL((thin_bp_batch_kernel<ZV, L>), dim3(blocks), dim3(64 * per_block),
                         (thin_bp_lds_bytes<ZV, L>(per_block)), s, t);
  });
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

}  // namespace vamx
