// Inclined projections (rays tilted by phi against the detector's rows) on
// wavefronts: forward of one ray, back projection of one voxel column, with z
// across the lanes.
//
// At inclination phi a sample at along-ray coordinate s lies s tan(phi)
// slices above the ray's detector row: floor q and fraction w of that shift
// are the same for every row, so a sample's in-plane taps, its absorption
// weight, q and w are wave-uniform.  Lane l evaluates the geometry of sample
// r0 + l (or angle i0 + l) once, in float64, into a per-wavefront LDS table;
// the wavefront then walks the table.  Lane l loads slice j + q of its
// detector row j and adds it, weighted 1 - w, to row j's sum and, weighted w,
// to a second sum that belongs to row j - 1 (whose upper slice it is): each
// in-plane tap is one load, not two.  The second sum moves down one lane
// after the walk, so the last lane's row is not complete and a wavefront
// covers 64 NS - 1 rows (L - 1 in the grouped form).  Slices outside the
// volume get an offset past the buffer descriptor's range and read 0.
//
// Below 64 rows (nz <= 31) the lanes form 64 / L groups of L; group g takes
// every (64 / L)-th table entry, and the groups' sums are added at the end.
//
// Bound by the texture path (forward): per sample and 64 rows four dword loads of
// 8.5 cycles each, and six multiply-adds; incl_fp_fixed_kernel loads fewer.  The per-lane
// kernels this replaces evaluated the float64 geometry in every lane and
// loaded eight taps per sample.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "par_core.h"

namespace vamx {

namespace {

constexpr int kU = 4;                 // table entries per step (loads in flight)
constexpr int kTab = 64 + kU * 8;     // entries past 64 are empty
constexpr int kNone = 1 << 29;        // shift of an empty entry: every slice is out of range, so it reads 0
constexpr int kOne = 1 << 28;         // cell flags: one column (kOne) or row (2 kOne) only -- the weightless
                                      // second one is not read (its voxels may lie outside, or hold no number)

struct InclSlot {
  float4* w;   // forward: bilinear tap weights; back: row weights for the two sums
  float4* a;   // forward: weights of the two sums, cell, shift; back: -, second row, row, shift
};
__device__ __forceinline__ InclSlot incl_slot() {
  __shared__ float4 w[4][kTab];
  __shared__ float4 a[4][kTab];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 3;
  return {w[wv], a[wv]};
}

__device__ __forceinline__ void incl_pad(const InclSlot& sl, int lane) {
  if (lane < kTab - 64) {
    sl.w[64 + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
    sl.a[64 + lane] = make_float4(0.f, 0.f, 0.f, __int_as_float(kNone));
  }
}

// the taps of one axis: first one b with weight s0, and b + 1 with s1 (0: no second tap)
__device__ __forceinline__ void axis_taps(double coord, int n, int& b, double& s0, double& s1) {
  const double f = floor(coord), d = coord - f;
  const int fi = (int)f;
  b = fi < 0 ? 0 : fi;
  s0 = fi < 0 ? d : 1.0 - d;
  s1 = fi < 0 || fi >= n - 1 ? 0.0 : d;
}

// byte offset of slice zz, or one that the descriptor's range rejects (reads 0)
__device__ __forceinline__ uint32_t slice_off(int zz, int nz) {
  return (unsigned)zz < (unsigned)nz ? 4u * (uint32_t)zz : 0x80000000u;
}

// completes the two sums of every row: out[s] is the row j0 + l + 64 s (valid
// below the wavefront's row count, in group 0)
template <int NS, int L>
__device__ __forceinline__ void incl_combine(float (&lo)[NS], float (&hi)[NS], int lane) {
  if constexpr (L < 64) {
#pragma unroll
    for (int o = L; o < 64; o <<= 1) {
      lo[0] += __shfl_xor(lo[0], o);
      hi[0] += __shfl_xor(hi[0], o);
    }
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    float up = __shfl_down(hi[s], 1);
    if (s + 1 < NS) {
      const float first = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hi[s + 1]), 0));
      if (lane == 63) up = first;
    }
    lo[s] += up;
  }
}

// rows of one wavefront
template <int NS, int L> constexpr int incl_rows() { return (L < 64 ? L : 64 * NS) - 1; }

// (lb in the functions of a block: its number in the problem)
template <int NS, int L, class Out>
__device__ __forceinline__ void incl_fp_block(const ParDev& g, const float* __restrict__ vol, const Out& out,
                                              unsigned lb) {
  constexpr int G = 64 / L, S = incl_rows<NS, L>();
  const int lane = threadIdx.x & 63, l = lane & (L - 1), grp = lane / L;
  const long long wave = wave_index(lb);
  const long long rays = (long long)g.n * g.na;
  const int nch = (g.nz + S - 1) / S;
  if (wave >= rays * nch) return;   // whole wavefronts
  const int j0 = (int)(wave / rays) * S;
  const int i = (int)((wave % rays) / g.n), k = (int)((wave % rays) % g.n);
  const int n = g.n, nz = g.nz;
  const double* M = g.mats + 6 * i;
  const double kp = (double)k - g.det_offset;
  const double a0 = M[0] * kp, a1 = M[3] * kp;
  const double t = (double)(k - g.c) - g.det_offset;
  const uint32_t oc = 4u * (uint32_t)nz, orr = (uint32_t)n * oc, span = orr + 2 * oc;
  const InclSlot sl = incl_slot();
  incl_pad(sl, lane);
  float lo[NS] = {}, hi[NS] = {};
  for (int r0 = 0; r0 < n; r0 += 64) {
    const int r = r0 + lane;
    float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
    float aw0 = 0.f, aw1 = 0.f;
    int base = 0, q = kNone;
    bool valid = false;
    if (r < n) {
      const double rr = (double)r;
      const double col = (a0 + M[1] * rr) + M[2];
      const double row = (a1 + M[4] * rr) + M[5];
      if (row > -1.0 && row < (double)n && col > -1.0 && col < (double)n) {
        int br, bc;
        double r0w, r1w, c0w, c1w;
        axis_taps(row, n, br, r0w, r1w);
        axis_taps(col, n, bc, c0w, c1w);
        const double s = (double)(r - g.c), dz = s * g.tan_phi, fz = floor(dz);
        const float aw = abs_weight(g, t, s);
        base = (br * n + bc) | (c1w == 0.0 ? kOne : 0) | (r1w == 0.0 ? 2 * kOne : 0);
        if (aw != 0.0f) q = (int)fz;
        aw0 = aw * (float)(1.0 - (dz - fz));
        aw1 = aw * (float)(dz - fz);
        w = make_float4((float)(r0w * c0w), (float)(r0w * c1w), (float)(r1w * c0w), (float)(r1w * c1w));
        valid = aw != 0.0f;
      }
    }
    const unsigned long long m = __ballot(valid);
    __builtin_amdgcn_wave_barrier();
    sl.w[lane] = w;
    sl.a[lane] = make_float4(aw0, aw1, __int_as_float(base), __int_as_float(q));
    __builtin_amdgcn_wave_barrier();
    if (!m) continue;
    const int first = __builtin_ctzll(m) & ~(G - 1), last = 63 - __builtin_clzll(m);
    for (int e0 = first; e0 <= last; e0 += kU * G) {
      float v[kU][NS][4];
      float4 ww[kU];
      float2 aa[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int e = e0 + u * G + grp;
        ww[u] = sl.w[e];
        const float4 A = sl.a[e];
        aa[u] = make_float2(A.x, A.y);
        const int b = __float_as_int(A.z), qs = __float_as_int(A.w);
        if constexpr (G == 1) {
          const int bu = __builtin_amdgcn_readfirstlane(b);
          const __amdgpu_buffer_rsrc_t rs = buf_rsrc(vol + (size_t)(bu & (kOne - 1)) * nz, span);
          const uint32_t o1 = bu & kOne ? 0u : oc, o2 = bu & (2 * kOne) ? 0u : orr;
          const int z = j0 + lane + __builtin_amdgcn_readfirstlane(qs);
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const uint32_t vo = slice_off(z + 64 * s, nz);
            v[u][s][0] = bload<1>(rs, vo, 0);
            v[u][s][1] = bload<1>(rs, vo, o1);
            v[u][s][2] = bload<1>(rs, vo, o2);
            v[u][s][3] = bload<1>(rs, vo, o1 + o2);
          }
        } else {
          const int z = j0 + l + qs;
          const bool in = (unsigned)z < (unsigned)nz;
          const float* p = vol + (size_t)(b & (kOne - 1)) * nz + (in ? z : 0);
          const int o1 = b & kOne ? 0 : nz, o2 = b & (2 * kOne) ? 0 : n * nz;
          const float x0 = p[0], x1 = p[o1], x2 = p[o2], x3 = p[o1 + o2];
          v[u][0][0] = in ? x0 : 0.0f;
          v[u][0][1] = in ? x1 : 0.0f;
          v[u][0][2] = in ? x2 : 0.0f;
          v[u][0][3] = in ? x3 : 0.0f;
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const float x = vfma(ww[u].w, v[u][s][3],
                               vfma(ww[u].z, v[u][s][2], vfma(ww[u].y, v[u][s][1], ww[u].x * v[u][s][0])));
          lo[s] = vfma(aa[u].x, x, lo[s]);
          hi[s] = vfma(aa[u].y, x, hi[s]);
        }
    }
  }
  incl_combine<NS, L>(lo, hi, lane);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int so = l + 64 * s;
    if (grp == 0 && so < S && j0 + so < nz) out.put(((size_t)k * g.na + i) * nz + j0 + so, lo[s]);
  }
}
template <int NS, int L, class Out>
__global__ __launch_bounds__(256) void incl_fp_kernel(ParDev g, const float* __restrict__ vol, Out out) {
  incl_fp_block<NS, L>(g, vol, out, xcd_remap(blockIdx.x, gridDim.x));
}
template <int NS, int L>
__global__ __launch_bounds__(256) void incl_fp_batch_kernel(LaneTable t) {
  unsigned lb;
  const int p = lane_problem(t, lb);
  incl_fp_block<NS, L>(t.items[p].g, t.in[p], StoreOut{t.out[p]}, lb);
}

// Forward of one ray where the shift over the whole ray is small against the
// lanes: lanes own fixed slices, so that a sample finds the taps it shares with
// the sample before (fp_ray_wave's scheme: two of four, as a rule) in registers,
// and the rows' sums move past the lanes instead, one lane up (down) each time the
// samples' shift grows (falls) by a slice.  A wavefront covers 64 NS slices from
// slice j0 + shift.lo on and completes the `rows` detector rows from j0 on, whose
// slices stay inside that range for every sample; slices outside the volume read 0.
//
// A tap of weight 0 is not read, and its register holds 0 then (it may lie outside,
// or hold no number).
//
// Bound by latency and instructions (two slices per lane: 4.6 4-byte loads and 30
// vector instructions per sample, against 8 loads and 24 with the rows' own lanes,
// which the texture path bound): 128 x 128 x 96 x 180, 12 degrees 279 -> 211 us (206
// with the sample's two slices multiplied into the ray's sum one after the other, which
// rounds it twice), x 256 x 90 398 -> 285, 100 x 100 x 300 x 60, 10 degrees 177 -> 121.
// values of the next / previous slice (lane, and across the NS registers); 0 past
// the ends
template <int NS>
__device__ __forceinline__ float slice_next(const float (&v)[NS], int s) {
  const int end = s + 1 < NS ? __builtin_amdgcn_readlane(__float_as_int(v[s + 1 < NS ? s + 1 : s]), 0) : 0;
  return __int_as_float(__builtin_amdgcn_update_dpp(end, __float_as_int(v[s]), 0x130 /* wave_shl:1 */, 0xf, 0xf, false));
}
template <int NS>
__device__ __forceinline__ float slice_prev(const float (&v)[NS], int s) {
  const int end = s > 0 ? __builtin_amdgcn_readlane(__float_as_int(v[s > 0 ? s - 1 : s]), 63) : 0;
  return __int_as_float(__builtin_amdgcn_update_dpp(end, __float_as_int(v[s]), 0x138 /* wave_shr:1 */, 0xf, 0xf, false));
}

template <int NS, class Out>
__device__ __forceinline__ void incl_fp_fixed_block(const ParDev& g, const float* __restrict__ vol,
                                                    const InclShift& shift, const Out& out, unsigned lb) {
  const int lane = threadIdx.x & 63;
  const long long wave = wave_index(lb);
  const long long rays = (long long)g.n * g.na;
  const int nch = (g.nz + shift.rows - 1) / shift.rows;
  if (wave >= rays * nch) return;   // whole wavefronts
  const int j0 = (int)(wave / rays) * shift.rows;
  const int i = (int)((wave % rays) / g.n), k = (int)((wave % rays) % g.n);
  const int n = g.n, nz = g.nz;
  const double* M = g.mats + 6 * i;
  const double kp = (double)k - g.det_offset;
  const double a0 = M[0] * kp, a1 = M[3] * kp;
  const double t = (double)(k - g.c) - g.det_offset;
  const uint32_t oc = 4u * (uint32_t)nz, orr = (uint32_t)n * oc;
  // tap offsets count from the first row the 64 samples reach, or (big) from the
  // sample's own cell; slices outside the volume lie past the descriptor's range
  const bool big = 66ull * orr + 2ull * oc >= 0x7fffffffull;
  const int z0 = j0 + shift.lo + lane;
  uint32_t zo[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) zo[s] = slice_off(z0 + 64 * s, nz);
  const InclSlot sl = incl_slot();
  float acc[NS] = {}, part[NS] = {}, T[4][NS] = {};   // T[2 a + b]: the tap of row parity a, column parity b
  auto add_part = [&]() {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      acc[s] += part[s];
      part[s] = 0.0f;
    }
  };
  int at = 0;                          // shift of the last sample walked: lane z holds row z - at
  bool any = false;
  int last = -1, last_need = 15;       // cell and needed taps of the sample before the 64 (-1: none)
  for (int r0 = 0; r0 < n; r0 += 64) {
    const int r = r0 + lane;
    float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
    float aw0 = 0.f, aw1 = 0.f;
    int br = 0, bc = 0, q = 0, need = 0;
    bool valid = false;
    if (r < n) {
      const double rr = (double)r;
      const double col = (a0 + M[1] * rr) + M[2];
      const double row = (a1 + M[4] * rr) + M[5];
      if (row > -1.0 && row < (double)n && col > -1.0 && col < (double)n) {
        double r0w, r1w, c0w, c1w;
        axis_taps(row, n, br, r0w, r1w);
        axis_taps(col, n, bc, c0w, c1w);
        const double s = (double)(r - g.c), dz = s * g.tan_phi, fz = floor(dz);
        const float aw = abs_weight(g, t, s);
        q = (int)fz;
        aw0 = aw * (float)(1.0 - (dz - fz));
        aw1 = aw * (float)(dz - fz);
        const float k00 = (float)(r0w * c0w), k01 = (float)(r0w * c1w), k10 = (float)(r1w * c0w), k11 = (float)(r1w * c1w);
        const bool pr = br & 1, pc = bc & 1;
        const float e0 = pc ? k01 : k00, e1 = pc ? k00 : k01, f0 = pc ? k11 : k10, f1 = pc ? k10 : k11;
        w = pr ? make_float4(f0, f1, e0, e1) : make_float4(e0, e1, f0, f1);
        need = (w.x != 0.0f) | (w.y != 0.0f) << 1 | (w.z != 0.0f) << 2 | (w.w != 0.0f) << 3;
        valid = aw != 0.0f;
      }
    }
    unsigned long long m = __ballot(valid);
    if (!m) {
      last = -1;
      continue;
    }
    const int cell = valid ? (br << 14) | bc : -1;   // n < 2^14
    const int upc = __shfl_up(cell, 1), upn = __shfl_up(need, 1);
    const int before = lane == 0 ? last : upc, held = lane == 0 ? last_need : upn;
    last = rl_i(cell, 63);
    last_need = rl_i(need, 63);
    const int dr = br - (before >> 14), dc = bc - (before & 0x3fff);
    // taps to load, and (bits 4 to 7) registers to clear
    int code = need | (15 & ~need) << 4;
    if (before >= 0) {
      int lacks = 15;
      if (dr >= -1 && dr <= 1 && dc >= -1 && dc <= 1)
        lacks = (dr ? 3 << (2 * ((br + (dr > 0)) & 1)) : 0) | (dc ? 5 << ((bc + (dc > 0)) & 1) : 0);
      code = (need & (lacks | ~held)) | (held & ~need) << 4;
    }
    const int row_lo = min(rl_i(br, __builtin_ctzll(m)), rl_i(br, 63 - __builtin_clzll(m)));
    const uint32_t from = big ? 0u : (uint32_t)(br - row_lo) * orr + (uint32_t)bc * oc;
    const uint32_t re = from + ((br & 1) ? orr : 0u), ro = from + ((br & 1) ? 0u : orr);
    const uint32_t ce = (bc & 1) ? oc : 0u, co = (bc & 1) ? 0u : oc;
    const int o00 = (int)(re + ce), o01 = (int)(re + co), o10 = (int)(ro + ce), o11 = (int)(ro + co);
    __amdgpu_buffer_rsrc_t rs = buf_rsrc(vol + (size_t)row_lo * n * nz, 0x7fffffffu);
    __builtin_amdgcn_wave_barrier();
    sl.w[lane] = w;
    sl.a[lane] = make_float4(aw0, aw1, 0.f, 0.f);
    __builtin_amdgcn_wave_barrier();
    // the samples are summed up to 16 at a time, as long as the shift stays: the
    // ray's sums are rounded once per part, not twice per sample
#pragma unroll 1
    for (int from = 0; from < 64; from += 16) {
      unsigned long long ms = m & (0xffffull << from);
      while (ms) {
        const int j = __builtin_ctzll(ms);
        ms &= ms - 1;
        const float4 W = sl.w[j], A = sl.a[j];
        const int c = rl_i(code, j), qj = rl_i(q, j);
        if (big) {
          const int b = rl_i(cell, j);
          rs = buf_rsrc(vol + ((size_t)(b >> 14) * n + (b & 0x3fff)) * nz, 0x7fffffffu);
        }
        auto tap = [&](int a, int o) {
          if (c >> a & 1) {
            const uint32_t so = (uint32_t)rl_i(o, j);
#pragma unroll
            for (int s = 0; s < NS; ++s) T[a][s] = bload<1>(rs, zo[s], so);
          }
        };
        tap(0, o00);
        tap(1, o01);
        tap(2, o10);
        tap(3, o11);
        if (c >> 4) {
#pragma unroll
          for (int a = 0; a < 4; ++a)
            if (c >> (4 + a) & 1)
#pragma unroll
              for (int s = 0; s < NS; ++s) T[a][s] = 0.0f;
        }
        if (!any) at = qj;   // nothing summed yet
        any = true;
        if (at != qj) add_part();
        while (at < qj) {
          float moved[NS];
#pragma unroll
          for (int s = 0; s < NS; ++s) moved[s] = slice_prev<NS>(acc, s);
#pragma unroll
          for (int s = 0; s < NS; ++s) acc[s] = moved[s];
          ++at;
        }
        while (at > qj) {
          float moved[NS];
#pragma unroll
          for (int s = 0; s < NS; ++s) moved[s] = slice_next<NS>(acc, s);
#pragma unroll
          for (int s = 0; s < NS; ++s) acc[s] = moved[s];
          --at;
        }
        float v[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s)
          v[s] = vfma(W.w, T[3][s], vfma(W.z, T[2][s], vfma(W.y, T[1][s], W.x * T[0][s])));
#pragma unroll
        for (int s = 0; s < NS; ++s) part[s] = vfma(A.y, slice_next<NS>(v, s), vfma(A.x, v[s], part[s]));
      }
      add_part();
    }
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int j = z0 + 64 * s - at;
    if (j >= j0 && j < j0 + shift.rows && j < nz) out.put(((size_t)k * g.na + i) * nz + j, acc[s]);
  }
}
template <int NS, class Out>
__global__ __launch_bounds__(256) void incl_fp_fixed_kernel(ParDev g, const float* __restrict__ vol, InclShift shift,
                                                            Out out) {
  incl_fp_fixed_block<NS>(g, vol, shift, out, xcd_remap(blockIdx.x, gridDim.x));
}
template <int NS>
__global__ __launch_bounds__(256) void incl_fp_fixed_batch_kernel(LaneTable t) {
  unsigned lb;
  const int p = lane_problem(t, lb);
  const LaneProblem& q = t.items[p];
  incl_fp_fixed_block<NS>(q.g, t.in[p], q.shift, StoreOut{t.out[p]}, lb);
}

template <int NS, int L>
__device__ __forceinline__ void incl_bp_block(const ParDev& g, const float* __restrict__ sino, float* __restrict__ vol,
                                              int clipc, unsigned lb) {
  constexpr int G = 64 / L, S = incl_rows<NS, L>();
  const int lane = threadIdx.x & 63, l = lane & (L - 1), grp = lane / L;
  const long long wave = wave_index(lb);
  // consecutive wavefronts walk 8 x 8 patches of voxel columns (neighbouring
  // columns read the same detector rows)
  const int n = g.n, nz = g.nz, nt = (n + 7) / 8;
  const long long cols = 64ll * nt * nt;
  const int nch = (nz + S - 1) / S;
  if (wave >= cols * nch) return;   // whole wavefronts
  const int j0 = (int)(wave / cols) * S;
  const int patch = (int)((wave % cols) >> 6), in = (int)(wave & 63);
  const int row = (patch / nt) * 8 + (in >> 3), col = (patch % nt) * 8 + (in & 7);
  if (row >= n || col >= n) return;
  float lo[NS] = {}, hi[NS] = {};
  if (!(clipc && g.outside[row * n + col])) {
    const double x = (double)(col - g.c), y = (double)(row - g.c);
    const uint32_t row_b = 4u * (uint32_t)g.na * (uint32_t)nz, span = row_b + 4u * (uint32_t)nz;
    const InclSlot sl = incl_slot();
    incl_pad(sl, lane);
    for (int i0 = 0; i0 < g.na; i0 += 64) {
      const int i = i0 + lane;
      float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
      int at = 0, q = kNone, step = 0;
      if (i < g.na) {
        const double co = g.cs[2 * i], sn = g.cs[2 * i + 1];
        const double t = x * co - y * sn;
        int j, j1;
        float f;
        if (interp_node(g, t, j, j1, f)) {
          const double s = x * sn + y * co, dz = -(s * g.tan_phi), fz = floor(dz);
          const float aw = abs_weight(g, t, s);
          const float b0 = aw * (float)(1.0 - (dz - fz)), b1 = aw * (float)(dz - fz);
          at = j * g.na + i;
          step = j1 > j;   // 0 exactly at the last node: fp[n - 1]
          if (aw != 0.0f) q = (int)fz;
          w = make_float4((1.0f - f) * b0, f * b0, (1.0f - f) * b1, f * b1);
        }
      }
      __builtin_amdgcn_wave_barrier();
      sl.w[lane] = w;
      sl.a[lane] = make_float4(0.f, __int_as_float(step), __int_as_float(at), __int_as_float(q));
      __builtin_amdgcn_wave_barrier();
      const int rows = g.na - i0 < 64 ? g.na - i0 : 64;
      for (int e0 = 0; e0 < rows; e0 += kU * G) {
        float v[kU][NS][2];
        float4 ww[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int e = e0 + u * G + grp;
          ww[u] = sl.w[e];
          const float4 A = sl.a[e];
          const int st = __float_as_int(A.y), b = __float_as_int(A.z), qs = __float_as_int(A.w);
          if constexpr (G == 1) {
            const uint32_t o1 = __builtin_amdgcn_readfirstlane(st) ? row_b : 0u;
            const __amdgpu_buffer_rsrc_t rs = buf_rsrc(sino + (size_t)__builtin_amdgcn_readfirstlane(b) * nz, span);
            const int z = j0 + lane + __builtin_amdgcn_readfirstlane(qs);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
              const uint32_t vo = slice_off(z + 64 * s, nz);
              v[u][s][0] = bload<1>(rs, vo, 0);
              v[u][s][1] = bload<1>(rs, vo, o1);
            }
          } else {
            const int z = j0 + l + qs;
            const bool in_z = (unsigned)z < (unsigned)nz;
            const float* p = sino + (size_t)b * nz + (in_z ? z : 0);
            const float x0 = p[0], x1 = p[st ? (size_t)g.na * nz : 0];
            v[u][0][0] = in_z ? x0 : 0.0f;
            v[u][0][1] = in_z ? x1 : 0.0f;
          }
        }
        // summed from zero and added once: the sums so far are rounded once a step
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          float pl = vfma(ww[0].y, v[0][s][1], ww[0].x * v[0][s][0]);
          float ph = vfma(ww[0].w, v[0][s][1], ww[0].z * v[0][s][0]);
#pragma unroll
          for (int u = 1; u < kU; ++u) {
            pl = vfma(ww[u].y, v[u][s][1], vfma(ww[u].x, v[u][s][0], pl));
            ph = vfma(ww[u].w, v[u][s][1], vfma(ww[u].z, v[u][s][0], ph));
          }
          lo[s] += pl;
          hi[s] += ph;
        }
      }
    }
    incl_combine<NS, L>(lo, hi, lane);
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int so = l + 64 * s;
    if (grp == 0 && so < S && j0 + so < nz) vol[((size_t)row * n + col) * nz + j0 + so] = lo[s];
  }
}
template <int NS, int L>
__global__ __launch_bounds__(256) void incl_bp_kernel(ParDev g, const float* __restrict__ sino,
                                                      float* __restrict__ vol, int clipc) {
  incl_bp_block<NS, L>(g, sino, vol, clipc, xcd_remap(blockIdx.x, gridDim.x));
}
template <int NS, int L>
__global__ __launch_bounds__(256) void incl_bp_batch_kernel(LaneTable t) {
  unsigned lb;
  const int p = lane_problem(t, lb);
  const LaneProblem& q = t.items[p];
  incl_bp_block<NS, L>(q.g, t.in[p], t.out[p], q.clip, lb);
}

// slabs of 64 rows per wavefront: a wavefront's geometry costs about 0.7 of a
// slab's walk, so NS minimises chunks (NS + 0.7)
int incl_slabs(int nz) {
  int best = 1;
  double cost = 1e30;
  for (int ns = 1; ns <= 3; ++ns) {
    const double c = (double)((nz + 64 * ns - 2) / (64 * ns - 1)) * (ns + 0.7);
    if (c < cost) {
      cost = c;
      best = ns;
    }
  }
  return best;
}

// slabs, and lanes of a row group, as slabs << 8 | lanes
int incl_layout(int nz) {
  if (nz <= 31) return 1 << 8 | (nz <= 7 ? 8 : nz <= 15 ? 16 : 32);
  return incl_slabs(nz) << 8 | 64;
}
template <class F>
void incl_dispatch(int layout, F&& f) {
  using std::integral_constant;
  if (layout == (1 << 8 | 8)) f(integral_constant<int, 1>{}, integral_constant<int, 8>{});
  else if (layout == (1 << 8 | 16)) f(integral_constant<int, 1>{}, integral_constant<int, 16>{});
  else if (layout == (1 << 8 | 32)) f(integral_constant<int, 1>{}, integral_constant<int, 32>{});
  else if (layout == (1 << 8 | 64)) f(integral_constant<int, 1>{}, integral_constant<int, 64>{});
  else if (layout == (2 << 8 | 64)) f(integral_constant<int, 2>{}, integral_constant<int, 64>{});
  else f(integral_constant<int, 3>{}, integral_constant<int, 64>{});
}
template <class F>
void incl_fixed_dispatch(int ns, F&& f) {
  using std::integral_constant;
  if (ns == 4) f(integral_constant<int, 4>{});
  else if (ns == 3) f(integral_constant<int, 3>{});
  else if (ns == 2) f(integral_constant<int, 2>{});
  else f(integral_constant<int, 1>{});
}
// wavefronts of a problem
long long incl_fixed_waves(const ParDev& g, const InclShift& shift) {
  return (long long)g.n * g.na * ((g.nz + shift.rows - 1) / shift.rows);
}
template <int NS, int L>
long long incl_fp_waves(const ParDev& g) {
  constexpr int S = incl_rows<NS, L>();
  return (long long)g.n * g.na * ((g.nz + S - 1) / S);
}
template <int NS, int L>
long long incl_bp_waves(const ParDev& g) {
  constexpr int S = incl_rows<NS, L>();
  const long long nt = (g.n + 7) / 8;
  return 64 * nt * nt * ((g.nz + S - 1) / S);
}

// whether the forward runs with fixed slices, and with how many slices per lane
// (0: with its own lanes' rows): the least time, by microseconds of a pass over 128
// x 128 columns, 180 angles, per chunk of rows -- 170, 200, 285, 370 with one to
// four fixed slices, of which the shift over a ray takes some lanes, and 150, 275,
// 400 with one to three rows (whose samples load all four taps and no shift is lost).
// Where both take one chunk of one register, rows win: 19 against 22 us at 64 x 64 x
// 48 x 60.  The figures are those of a GPU that is full; of 24 x 24 to 100 x 100 columns,
// where it is not, no size was found slower than by one thread per row.
int incl_fixed(const ParDev& g, InclShift& shift) {
  if (g.nz < 32) return 0;
  const double e0 = -(double)g.c * g.tan_phi, e1 = (double)(g.n - 1 - g.c) * g.tan_phi;
  const double lo = std::floor(std::min(e0, e1)), span = std::floor(std::max(e0, e1)) - lo;
  constexpr int fixed_us[5] = {0, 170, 200, 285, 370}, rows_us[4] = {0, 150, 275, 400};
  const int slabs = incl_slabs(g.nz), own = 64 * slabs - 1;
  long long best = (long long)((g.nz + own - 1) / own) * rows_us[slabs];
  int ns = 0;
  for (int k = 1; k <= 4; ++k) {
    if (span > 64 * k - 2) continue;
    const int rows = 64 * k - 1 - (int)span;
    const long long t = (long long)((g.nz + rows - 1) / rows) * fixed_us[k];
    if (t >= best) continue;
    best = t;
    ns = k;
    shift = {(int)lo, rows};
  }
  return ns;
}

template <class Out>
int incl_forward(vamx_plan* p, const float* vol, Out out, hipStream_t s) {
  const ParDev& g = p->par;
  InclShift shift;
  if (const int fixed = incl_fixed(g, shift)) {
    incl_fixed_dispatch(fixed, [&](auto ns) {
      hipLaunchKernelGGL((incl_fp_fixed_kernel<decltype(ns)::value, Out>),
                         dim3(blocks_for(incl_fixed_waves(g, shift) * 64, 256)), dim3(256), 0, s, g, vol, shift, out);
    });
  } else {
    incl_dispatch(incl_layout(g.nz), [&](auto ns, auto l) {
      constexpr int NS = decltype(ns)::value, L = decltype(l)::value;
      const dim3 grid(blocks_for(incl_fp_waves<NS, L>(g) * 64, 256));
      hipLaunchKernelGGL((incl_fp_kernel<NS, L, Out>), grid, dim3(256), 0, s, g, vol, out);
    });
  }
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

}  // namespace

bool incl_wave_ok(const vamx_plan* p) {
  return p->par.incl && p->par.n >= 2 && !(p->flags & VAMX_PAR_PER_LANE_GEOMETRY);
}

int incl_forward_store(vamx_plan* p, const float* vol, float* sino, hipStream_t s) {
  return incl_forward(p, vol, StoreOut{sino}, s);
}

int incl_forward_update(vamx_plan* p, const float* vol, const UpdateOut& out, hipStream_t s) {
  return incl_forward(p, vol, out, s);
}

int incl_backward(vamx_plan* p, const float* sino, float* vol, bool clipc, hipStream_t s) {
  const ParDev& g = p->par;
  incl_dispatch(incl_layout(g.nz), [&](auto ns, auto l) {
    constexpr int NS = decltype(ns)::value, L = decltype(l)::value;
    const dim3 grid(blocks_for(incl_bp_waves<NS, L>(g) * 64, 256));
    hipLaunchKernelGGL((incl_bp_kernel<NS, L>), grid, dim3(256), 0, s, g, sino, vol, clipc ? 1 : 0);
  });
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

// class of a problem: 2 << 16, 1 << 15 forward, then fixed slices 1 << 14 | slices
// per lane, or incl_layout
LaneClass incl_class(const vamx_plan* p, bool forward, bool clip) {
  const ParDev& g = p->par;
  LaneClass c;
  if (!incl_wave_ok(p)) return c;
  c.problem.g = g;
  c.problem.clip = clip;
  const int fixed = forward ? incl_fixed(g, c.problem.shift) : 0, layout = incl_layout(g.nz);
  if (fixed) {
    c.waves = incl_fixed_waves(g, c.problem.shift);
  } else {
    incl_dispatch(layout, [&](auto ns, auto l) {
      constexpr int NS = decltype(ns)::value, L = decltype(l)::value;
      c.waves = forward ? incl_fp_waves<NS, L>(g) : incl_bp_waves<NS, L>(g);
    });
  }
  c.blocks = (c.waves + 3) / 4;
  c.key = 2 << 16 | (forward ? 1 << 15 : 0) | (fixed ? 1 << 14 | fixed : layout);
  return c;
}

int incl_batch(int key, const LaneTable& t, unsigned blocks, hipStream_t s) {
  const dim3 grid(blocks), block(256);
  if (key >> 14 & 1) {
    incl_fixed_dispatch(key & 7, [&](auto ns) {
      hipLaunchKernelGGL((incl_fp_fixed_batch_kernel<decltype(ns)::value>), grid, block, 0, s, t);
    });
  } else {
    incl_dispatch(key & 0x3fff, [&](auto ns, auto l) {
      constexpr int NS = decltype(ns)::value, L = decltype(l)::value;
      if (key >> 15 & 1) hipLaunchKernelGGL((incl_fp_batch_kernel<NS, L>), grid, block, 0, s, t);
      else hipLaunchKernelGGL((incl_bp_batch_kernel<NS, L>), grid, block, 0, s, t);
    });
  }
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

}  // namespace vamx
