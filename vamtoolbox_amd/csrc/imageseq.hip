// Image-sequence export for gfx950: the frames a DLP projector shows, one per
// angle, composed from the sinogram on the device.
//
// Reference: vamtoolbox/imagesequence.py, ImageSeq.__init__ (85-182) and its
// helpers (300-399):
//   flips of the u / v axes, rotation in the (u, v) plane
//   (scipy.ndimage.rotate, order 1, reshape=True, constant 0 outside),
//   size scaling (OpenCV resize, INTER_LINEAR), percentile normalisation,
//   intensity scale, truncation at 2^bit_depth - 1, cast to the bit depth's
//   unsigned type, and insertion of one or more copies of each angle's
//   (v, u) image into a zeroed uint8 frame (a later copy overwrites an earlier
//   one; wider types wrap modulo 256 on insertion, as NumPy's assignment does).
//
// Three kernels, all float64 like the reference's NumPy arrays:
//   imgseq_rotate   one thread per output sample (v fastest), flips fused into
//                   the read;
//   imgseq_resize   one thread per output sample, flips fused into the read;
//   imgseq_compose  one 256-thread block per 64 x 64 tile of one angle's
//                   image: the tile's samples are read along v (the sinogram's
//                   fastest axis, coalesced), converted to bytes, transposed
//                   through LDS and written along u (the frame's fastest axis)
//                   into every copy.
#include <algorithm>

#include "vamx_internal.h"

namespace vamx {

namespace {

// scipy's order-1 affine transform in 'constant' mode: a sample whose
// coordinate lies outside [0, n - 1] on either axis is 0; inside, the four
// neighbours are summed as ((v * wy) * wx) in (0,0), (0,1), (1,0), (1,1)
// order, a neighbour beyond the last row / column counting as 0.
__global__ __launch_bounds__(256) void imgseq_rotate(const double* __restrict__ in, long long nu, long long na,
                                                     long long nv, int flip_u, int flip_v, double m00, double m01,
                                                     double m10, double m11, double off0, double off1,
                                                     double* __restrict__ out, long long mu, long long mv) {
#pragma clang fp contract(off)
  const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= mu * na * mv) return;
  const long long k = tid % mv;
  const long long j = (tid / mv) % na;
  const long long i = tid / (mv * na);
  const double fi = (double)i, fk = (double)k;
  const double cy = m00 * fi + m01 * fk + off0;
  const double cx = m10 * fi + m11 * fk + off1;
  double v = 0.0;
  if (cy >= 0.0 && cy <= (double)(nu - 1) && cx >= 0.0 && cx <= (double)(nv - 1)) {
    const double y0f = floor(cy), x0f = floor(cx);
    const double ty = cy - y0f, tx = cx - x0f;
    const long long y0 = (long long)y0f, x0 = (long long)x0f;
    const double wy[2] = {1.0 - ty, ty}, wx[2] = {1.0 - tx, tx};
    double t = 0.0;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const long long yy = y0 + a, xx = x0 + b;
        double s = 0.0;
        if (yy < nu && xx < nv) {
          const long long ys = flip_u ? nu - 1 - yy : yy, xs = flip_v ? nv - 1 - xx : xx;
          s = in[(ys * na + j) * nv + xs];
        }
        t += (s * wy[a]) * wx[b];
      }
    }
    v = t;
  }
  out[tid] = v;
}

// OpenCV INTER_LINEAR: destination index d samples (d + 0.5) * (src / dst) -
// 0.5; the integer part is clamped to [0, src - 1] with a zero fraction at
// either edge.
__device__ __forceinline__ void linear_tap(long long d, long long n_src, long long n_dst, long long& i0,
                                           long long& i1, double& t) {
#pragma clang fp contract(off)
  const double f = ((double)d + 0.5) * ((double)n_src / (double)n_dst) - 0.5;
  const double f0 = floor(f);
  i0 = (long long)f0;
  t = f - f0;
  if (i0 < 0) {
    t = 0.0;
    i0 = 0;
  }
  if (i0 >= n_src - 1) {
    t = 0.0;
    i0 = n_src - 1;
  }
  i1 = i0 + 1 < n_src ? i0 + 1 : n_src - 1;
}

__global__ __launch_bounds__(256) void imgseq_resize(const double* __restrict__ in, long long nu, long long na,
                                                     long long nv, int flip_u, int flip_v, double* __restrict__ out,
                                                     long long mu, long long mv) {
#pragma clang fp contract(off)
  const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= mu * na * mv) return;
  const long long k = tid % mv;
  const long long j = (tid / mv) % na;
  const long long i = tid / (mv * na);
  long long y0, y1, x0, x1;
  double ty, tx;
  linear_tap(i, nu, mu, y0, y1, ty);
  linear_tap(k, nv, mv, x0, x1, tx);
  auto at = [&](long long y, long long x) {
    const long long ys = flip_u ? nu - 1 - y : y, xs = flip_v ? nv - 1 - x : x;
    return in[(ys * na + j) * nv + xs];
  };
  const double top = at(y0, x0) * (1.0 - tx) + at(y0, x1) * tx;
  const double bot = at(y1, x0) * (1.0 - tx) + at(y1, x1) * tx;
  out[tid] = top * (1.0 - ty) + bot * ty;
}

constexpr int kTile = 64;
constexpr int kPitch = 68;   // bytes per LDS row: 17 dwords, so 64 lanes writing one column hit 64 banks

struct ComposeDev {
  int n_u, n_v, u1, n_copies, bit_depth, normalize, flip_u, flip_v;
  int tile_u0;   // first column tile of the launch
  int wide;      // rows of 16-byte stores
  double norm_value, max_value, intensity_scale;
  int v1[VAMX_IMGSEQ_MAX_COPIES];
};

// truncate at max_value (NaN passes, as np.minimum), cast toward zero to the
// unsigned type (NaN and negatives give 0), keep the low byte
__device__ __forceinline__ unsigned char to_byte(const ComposeDev& d, double x) {
#pragma clang fp contract(off)
  if (d.normalize) x = x / d.norm_value * d.max_value;
  if (d.intensity_scale != 1.0) x = x * d.intensity_scale;
  if (x > d.max_value) x = d.max_value;
  if (!(x >= 0.0)) return 0;
  return (unsigned char)((unsigned)x & 0xffu);
}

// zero frames: 16-byte stores (WIDE) or dword stores, grid-stride
template <bool WIDE>
__global__ __launch_bounds__(256) void imgseq_clear(unsigned char* __restrict__ frames, long long nbytes) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  if (WIDE) {
    uint4* f = reinterpret_cast<uint4*>(frames);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < nbytes / 16; i += stride)
      f[i] = make_uint4(0u, 0u, 0u, 0u);
  } else {
    unsigned* f = reinterpret_cast<unsigned*>(frames);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < nbytes / 4; i += stride) f[i] = 0u;
  }
}

// One block: the image rows of a 64-row tile times the 64 frame columns of a tile.
// Bound by memory: the image is read once (8 bytes a sample), while the zeros that
// imgseq_clear left in the caches drain.  A lane has its 16 samples in flight
// before the first is converted, and a sample is read and converted once for all
// copies.  256 x 256 x 360 (189 MB) in two copies into 1920 x 1080 frames: 157 ->
// 108 us (a block per frame tile, one sample at a time -> this), with the 127 us of
// the 746 MB of zeros 4.2 TB/s.  Tiles of 128 rows, 1 KiB runs: 108 us too.
__global__ __launch_bounds__(256) void imgseq_compose(ComposeDev d, const double* __restrict__ img, long long mu,
                                                      long long na, long long mv, unsigned char* __restrict__ frames) {
  __shared__ __align__(16) unsigned char tile[kTile * kPitch];
  const int u0 = (d.tile_u0 + (int)blockIdx.x) * kTile, r0 = (int)blockIdx.y * kTile;
  const long long j = blockIdx.z;
  const int t = threadIdx.x;
  // load: lanes along v (the image's contiguous axis), 4 columns per pass
  {
    const int rl = t & 63;
    const bool row = r0 + rl < (int)mv;
    const long long rs = d.flip_v ? mv - 1 - (r0 + rl) : r0 + rl;
    double x[kTile / 4];
#pragma unroll
    for (int q = 0; q < kTile / 4; ++q) {
      const int c = u0 + (t >> 6) + 4 * q - d.u1;
      x[q] = -1.0;   // outside the image: byte 0
      if (row && c >= 0 && c < (int)mu) x[q] = img[((d.flip_u ? mu - 1 - c : c) * na + j) * mv + rs];
    }
#pragma unroll
    for (int q = 0; q < kTile / 4; ++q) {
      const int ul = (t >> 6) + 4 * q, c = u0 + ul - d.u1;
      tile[rl * kPitch + ul] = row && c >= 0 && c < (int)mu ? to_byte(d, x[q]) : 0;
    }
  }
  __syncthreads();
  // store: 4 threads per row of every copy, 16 bytes each
  const int rl = t >> 2, ch = t & 3;
  if (r0 + rl >= (int)mv) return;
  const unsigned* src = reinterpret_cast<const unsigned*>(tile + rl * kPitch + ch * 16);
  const unsigned w[4] = {src[0], src[1], src[2], src[3]};
  const int u = u0 + ch * 16;
  for (int c = 0; c < d.n_copies; ++c) {
    const int v = d.v1[c] + r0 + rl;
    bool last = true;   // a later copy covering the row wins
    for (int k = c + 1; k < d.n_copies; ++k)
      if (v >= d.v1[k] && v < d.v1[k] + (int)mv) last = false;
    if (!last) continue;
    unsigned char* at = frames + ((size_t)j * d.n_v + v) * d.n_u + u;
    if (d.wide) {
      if (u < d.n_u) *reinterpret_cast<uint4*>(at) = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (u + q * 4 + 4 <= d.n_u) *reinterpret_cast<unsigned*>(at + q * 4) = w[q];
    }
  }
}

// ---------------------------------------------------------------------------
// Order statistics for np.percentile (imagesequence.py:128-131): the values
// of rank r and r + 1 of a float64 array, exactly, by radix selection on 64-bit
// keys whose unsigned order is the numeric order.  Pass p histograms digit p (12
// bits, most significant first; the last has 4) of the elements whose higher
// digits equal the ones selected so far.  Every block of a launch first picks the
// bucket of the previous pass that holds the rank (its histogram is complete) and
// so has the digits and the rank within them.  The counts are integers: the
// result is exact and does not depend on the launch.
//
// Two passes leave the elements that share 24 bits with the answer, a few
// thousand of 10^7 smoothly distributed ones: one more pass lists them (and takes
// the least key above them), and one block selects from the list.  The remaining
// passes run only where they are more than the list holds (many equal values);
// arrays the list holds as a whole are listed at once.
// Bound by reading the array: 23.6 M elements (189 MB) 39 us for a histogram pass
// (4.9 TB/s) and 31 us for the listing one, all in all 152 us; the eight passes of
// 8 bits, each with its own selection launch, and one for the key above took 362.
// ---------------------------------------------------------------------------
constexpr int OS_PASSES = 6, OS_BITS = 12, OS_BINS = 1 << OS_BITS;
constexpr int OS_LIST = 32768;
constexpr int OS_THREADS = 1024;
struct OsWork {
  unsigned long long counts[OS_PASSES][OS_BINS];
  unsigned long long prefix[OS_PASSES + 1];   // digits selected before pass p
  unsigned long long rem[OS_PASSES + 1];      // rank within the elements matching them
  unsigned long long bucket[OS_PASSES + 1];   // elements matching them
  unsigned long long nans;     // NaN elements
  unsigned long long min_gt;   // least key above the listed ones, or above the rank-r key
  unsigned long long listed;   // elements in list
  unsigned long long list[OS_LIST];
};
__host__ __device__ constexpr int os_shift(int pass) { return pass < 5 ? 52 - 12 * pass : 0; }
__host__ __device__ constexpr unsigned os_mask(int pass) { return pass < 5 ? 4095u : 15u; }

// negative values bit-inverted, others with the sign bit set: -0 sorts just
// below +0, NaN beyond -inf / +inf (a NaN anywhere makes the result NaN)
__device__ __forceinline__ unsigned long long os_key(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ __forceinline__ double os_value(unsigned long long k) {
  const unsigned long long b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
  return __longlong_as_double((long long)b);
}

__global__ __launch_bounds__(256) void os_init(OsWork* w, long long rank, long long n) {
  unsigned long long* c = &w->counts[0][0];
  for (int i = blockIdx.x * 256 + threadIdx.x; i < OS_PASSES * OS_BINS; i += 256 * gridDim.x) c[i] = 0ull;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    w->prefix[0] = 0ull;
    w->rem[0] = (unsigned long long)rank;
    w->bucket[0] = (unsigned long long)n;
    w->nans = 0ull;
    w->min_gt = ~0ull;
    w->listed = 0ull;
  }
}

struct OsPick {
  unsigned long long prefix, rem, bucket;
};

// inclusive sums over the block's OS_THREADS values
__device__ __forceinline__ unsigned long long os_scan(unsigned long long v, unsigned long long* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long u = __shfl_up(v, o);
    if (lane >= o) v += u;
  }
  __syncthreads();
  if (lane == 63) sh[wave] = v;
  __syncthreads();
  for (int k = 0; k < wave; ++k) v += sh[k];
  return v;
}

// the bucket of pass `pass`'s complete histogram that holds the rank; the first
// block leaves it for the next launch
__device__ __forceinline__ OsPick os_pick(OsWork* w, int pass) {
  __shared__ unsigned long long sh[OS_THREADS / 64];
  __shared__ OsPick found;
  const int t = threadIdx.x;
  const unsigned long long rem = w->rem[pass];
  unsigned long long c[OS_BINS / OS_THREADS], sum = 0ull;
#pragma unroll
  for (int q = 0; q < OS_BINS / OS_THREADS; ++q) {
    c[q] = w->counts[pass][t * (OS_BINS / OS_THREADS) + q];
    sum += c[q];
  }
  unsigned long long at = os_scan(sum, sh) - sum;
#pragma unroll
  for (int q = 0; q < OS_BINS / OS_THREADS; ++q) {
    if (at <= rem && rem < at + c[q]) {   // exactly one digit
      const unsigned long long digit = t * (OS_BINS / OS_THREADS) + q;
      found = {w->prefix[pass] | (digit << os_shift(pass)), rem - at, c[q]};
    }
    at += c[q];
  }
  __syncthreads();
  const OsPick p = found;
  if (blockIdx.x == 0 && t == 0) {
    w->prefix[pass + 1] = p.prefix;
    w->rem[pass + 1] = p.rem;
    w->bucket[pass + 1] = p.bucket;
  }
  return p;
}

// calls f(value) for every element; a lane's loads of a turn are issued together
template <bool VEC, class F>
__device__ __forceinline__ void os_each(const double* __restrict__ x, long long n, F&& f) {
  const long long gid = (long long)blockIdx.x * OS_THREADS + threadIdx.x, stride = (long long)gridDim.x * OS_THREADS;
  if (VEC) {
    const double2* x2 = reinterpret_cast<const double2*>(x);
    const long long m = n / 2;
    for (long long i = gid; i < m; i += 4 * stride) {
      double2 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = x2[i + q * stride < m ? i + q * stride : i];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (i + q * stride >= m) break;
        f(v[q].x);
        f(v[q].y);
      }
    }
    if (gid == 0 && (n & 1)) f(x[n - 1]);
  } else {
    for (long long i = gid; i < n; i += stride) f(x[i]);
  }
}

// adds a digit to the block histogram when its higher digits match; lanes
// sharing the first active lane's digit add once, together
__device__ __forceinline__ void os_count(unsigned* h, bool match, unsigned d) {
  const unsigned lead = __builtin_amdgcn_readfirstlane(match ? d : ~0u);
  const unsigned long long same = __ballot(match && d == lead);
  if (match && d == lead) {
    if (__lane_id() == (unsigned)__ffsll((long long)same) - 1u) atomicAdd(&h[d], (unsigned)__popcll(same));
  } else if (match) {
    atomicAdd(&h[d], 1u);
  }
}

// pass PASS's histogram; from pass 2 on only where the list does not do
template <bool VEC>
__global__ __launch_bounds__(OS_THREADS) void os_hist(const double* __restrict__ x, long long n, OsWork* w, int pass) {
  __shared__ unsigned h[OS_BINS];
  if (pass >= 2 && w->bucket[2] <= (unsigned long long)OS_LIST) return;   // grid-uniform
  const int t = threadIdx.x;
  for (int i = t; i < OS_BINS; i += OS_THREADS) h[i] = 0u;
  const unsigned long long prefix = pass ? os_pick(w, pass - 1).prefix : 0ull;
  __syncthreads();
  const int shift = os_shift(pass), above = pass < 5 ? shift + 12 : 4;
  const unsigned mask = os_mask(pass);
  unsigned long long nan_count = 0ull;
  os_each<VEC>(x, n, [&](double v) {
    if (pass == 0 && v != v) ++nan_count;
    const unsigned long long k = os_key(v);
    os_count(h, pass == 0 || (k >> above) == (prefix >> above), (unsigned)(k >> shift) & mask);
  });
  if (nan_count) atomicAdd(&w->nans, nan_count);
  __syncthreads();
  for (int i = t; i < OS_BINS; i += OS_THREADS)
    if (h[i]) atomicAdd(&w->counts[pass][i], (unsigned long long)h[i]);
}

// least key of the block's lanes into w->min_gt; every thread of the block takes
// part.  One atomic per block: with one per wavefront the 8192 minima at the one
// address took longer than the array's reading where values above the rank are
// spread over all wavefronts: os_collect over 23.6 M uniform values 121 -> 36 us, over
// the projections of a part 50 -> 31 us (6.0 TB/s).
__device__ __forceinline__ void os_min(unsigned long long m, OsWork* w) {
  __shared__ unsigned long long sh[OS_THREADS / 64];
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long q = __shfl_xor(m, o);
    m = q < m ? q : m;
  }
  if (__lane_id() == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < OS_THREADS / 64; ++k) m = sh[k] < m ? sh[k] : m;
    if (m != ~0ull) atomicMin(&w->min_gt, m);
  }
}

// the bucket's count bounds the list; the test keeps calls that wrongly share a
// workspace inside it
__device__ __forceinline__ void os_put(OsWork* w, unsigned long long at, unsigned long long k) {
  if (at < (unsigned long long)OS_LIST) w->list[at] = k;
}

// lists the elements that share the first two digits with the answer, through
// LDS (one addition to the list's length per block), and takes the least key
// above them
template <bool VEC>
__global__ __launch_bounds__(OS_THREADS) void os_collect(const double* __restrict__ x, long long n, OsWork* w) {
  __shared__ unsigned long long buf[1024], base;
  __shared__ unsigned held;
  if (threadIdx.x == 0) held = 0u;
  const OsPick p = os_pick(w, 1);
  if (p.bucket > (unsigned long long)OS_LIST) return;   // grid-uniform
  unsigned long long m = ~0ull;
  os_each<VEC>(x, n, [&](double v) {
    const unsigned long long k = os_key(v);
    if ((k >> 40) == (p.prefix >> 40)) {
      const unsigned at = atomicAdd(&held, 1u);
      if (at < 1024u) buf[at] = k;
      else os_put(w, atomicAdd(&w->listed, 1ull), k);
    } else if (k > p.prefix && k < m) {
      m = k;
    }
  });
  os_min(m, w);
  __syncthreads();
  const unsigned c = held < 1024u ? held : 1024u;
  if (threadIdx.x == 0 && c) base = atomicAdd(&w->listed, (unsigned long long)c);
  __syncthreads();
  if (threadIdx.x < c) os_put(w, base + threadIdx.x, buf[threadIdx.x]);
}

// lists a whole array of at most OS_LIST elements
__global__ __launch_bounds__(OS_THREADS) void os_list(const double* __restrict__ x, long long n, OsWork* w) {
  const long long i = (long long)blockIdx.x * OS_THREADS + threadIdx.x;
  if (i == 0) w->listed = (unsigned long long)n;
  if (i >= n) return;
  const double v = x[i];
  if (v != v) atomicAdd(&w->nans, 1ull);
  w->list[i] = os_key(v);
}

// least key above the rank-r key, where all passes ran
template <bool VEC>
__global__ __launch_bounds__(OS_THREADS) void os_tail(const double* __restrict__ x, long long n, OsWork* w) {
  if (w->bucket[2] <= (unsigned long long)OS_LIST) return;   // grid-uniform
  const OsPick p = os_pick(w, OS_PASSES - 1);
  if (p.rem + 1 < p.bucket) return;   // rank r + 1 holds an equal key
  unsigned long long m = ~0ull;
  os_each<VEC>(x, n, [&](double v) {
    const unsigned long long k = os_key(v);
    if (k > p.prefix && k < m) m = k;
  });
  os_min(m, w);
}

// one block: the values of ranks r and r + 1, from the list by 8-bit digits where
// it holds them (all: it holds every element)
__global__ __launch_bounds__(OS_THREADS) void os_finish(long long n, long long rank, int all, OsWork* w, double* out) {
  __shared__ unsigned h[256];
  __shared__ unsigned long long sh[OS_THREADS / 64];
  __shared__ unsigned long long s_key, s_rem, s_next;
  const int t = threadIdx.x;
  unsigned long long key = w->prefix[OS_PASSES], rem = w->rem[OS_PASSES], count = w->bucket[OS_PASSES];
  if (all || w->bucket[2] <= (unsigned long long)OS_LIST) {
    const int listed = (int)(w->listed < (unsigned long long)OS_LIST ? w->listed : (unsigned long long)OS_LIST);
    key = all ? 0ull : w->prefix[2];
    rem = all ? (unsigned long long)rank : w->rem[2];
    for (int shift = all ? 56 : 32; shift >= 0; shift -= 8) {
      if (t < 256) h[t] = 0u;
      __syncthreads();
      for (int i = t; i < listed; i += OS_THREADS) {
        const unsigned long long k = w->list[i];
        if (shift == 56 || (k >> (shift + 8)) == (key >> (shift + 8))) atomicAdd(&h[(k >> shift) & 255u], 1u);
      }
      __syncthreads();
      const unsigned long long c = t < 256 ? h[t] : 0u, incl = os_scan(c, sh);
      if (incl - c <= rem && rem < incl) {   // exactly one digit
        s_key = key | ((unsigned long long)t << shift);
        s_rem = rem - (incl - c);
      }
      __syncthreads();
      key = s_key;
      rem = s_rem;
      count = h[(key >> shift) & 255u];
      __syncthreads();
    }
    if (t == 0) s_next = w->min_gt;
    __syncthreads();
    for (int i = t; i < listed; i += OS_THREADS) {
      const unsigned long long k = w->list[i];
      if (k > key) atomicMin(&s_next, k);
    }
    __syncthreads();
  } else if (t == 0) {
    s_next = w->min_gt;
  }
  if (t != 0) return;
  const double a = os_value(key);
  const double b = rank + 1 < n && rem + 1 >= count ? os_value(s_next) : a;
  const double nan = __longlong_as_double(0x7ff8000000000000ll);
  out[0] = w->nans ? nan : a;
  out[1] = w->nans ? nan : b;
}

}  // namespace

}  // namespace vamx

using namespace vamx;

extern "C" int vamx_order_stats_workspace_bytes(int64_t* bytes) {
  if (!bytes) return set_error(VAMX_ERR_ARG, "vamx_order_stats_workspace_bytes: null argument");
  *bytes = (int64_t)sizeof(OsWork);
  return VAMX_OK;
}

extern "C" int vamx_order_stats(const double* x, int64_t n, int64_t rank, double* out, void* workspace,
                                void* stream) {
  if (!x || !out || !workspace) return set_error(VAMX_ERR_ARG, "vamx_order_stats: null argument");
  if (n < 1) return set_error(VAMX_ERR_ARG, "vamx_order_stats: empty array");
  if (rank < 0 || rank >= n) return set_error(VAMX_ERR_ARG, "vamx_order_stats: rank outside 0 .. n-1");
  if ((uintptr_t)workspace % 8) return set_error(VAMX_ERR_ARG, "vamx_order_stats: workspace must be 8-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  OsWork* w = (OsWork*)workspace;
  // two blocks of 1024 threads per CU
  const dim3 grid((unsigned)std::min<long long>(512, (n + 2 * OS_THREADS - 1) / (2 * OS_THREADS))), block(OS_THREADS);
  const bool vec = (uintptr_t)x % 16 == 0;
  const int all = n <= OS_LIST ? 1 : 0;
  hipLaunchKernelGGL(os_init, dim3(all ? 1 : 24), dim3(256), 0, s, w, (long long)rank, (long long)n);
  auto launch = [&](auto kernel_vec, auto kernel, auto... args) {
    if (vec) hipLaunchKernelGGL(kernel_vec, grid, block, 0, s, x, (long long)n, w, args...);
    else hipLaunchKernelGGL(kernel, grid, block, 0, s, x, (long long)n, w, args...);
  };
  if (all) {
    hipLaunchKernelGGL(os_list, dim3((unsigned)((n + OS_THREADS - 1) / OS_THREADS)), block, 0, s, x, (long long)n, w);
  } else {
    for (int p = 0; p < 2; ++p) launch(os_hist<true>, os_hist<false>, p);
    launch(os_collect<true>, os_collect<false>);
    for (int p = 2; p < OS_PASSES; ++p) launch(os_hist<true>, os_hist<false>, p);
    launch(os_tail<true>, os_tail<false>);
  }
  hipLaunchKernelGGL(os_finish, dim3(1), block, 0, s, (long long)n, (long long)rank, all, w, out);
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

extern "C" int vamx_imgseq_rotate(const double* in, int64_t nu, int64_t na, int64_t nv, int32_t flip_u,
                                  int32_t flip_v, const double* matrix, const double* offset, double* out,
                                  int64_t mu, int64_t mv, void* stream) {
  if (!in || !out || !matrix || !offset) return set_error(VAMX_ERR_ARG, "vamx_imgseq_rotate: null argument");
  if (nu < 1 || na < 1 || nv < 1 || mu < 1 || mv < 1)
    return set_error(VAMX_ERR_ARG, "vamx_imgseq_rotate: empty array");
  hipLaunchKernelGGL(imgseq_rotate, dim3(blocks_for(mu * na * mv, 256)), dim3(256), 0, (hipStream_t)stream, in,
                     (long long)nu, (long long)na, (long long)nv, flip_u ? 1 : 0, flip_v ? 1 : 0, matrix[0],
                     matrix[1], matrix[2], matrix[3], offset[0], offset[1], out, (long long)mu, (long long)mv);
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

extern "C" int vamx_imgseq_resize(const double* in, int64_t nu, int64_t na, int64_t nv, int32_t flip_u,
                                  int32_t flip_v, double* out, int64_t mu, int64_t mv, void* stream) {
  if (!in || !out) return set_error(VAMX_ERR_ARG, "vamx_imgseq_resize: null argument");
  if (nu < 1 || na < 1 || nv < 1 || mu < 1 || mv < 1)
    return set_error(VAMX_ERR_ARG, "vamx_imgseq_resize: empty array");
  hipLaunchKernelGGL(imgseq_resize, dim3(blocks_for(mu * na * mv, 256)), dim3(256), 0, (hipStream_t)stream, in,
                     (long long)nu, (long long)na, (long long)nv, flip_u ? 1 : 0, flip_v ? 1 : 0, out,
                     (long long)mu, (long long)mv);
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}

extern "C" int vamx_imgseq_compose(const double* img, int64_t mu, int64_t na, int64_t mv,
                                   const vamx_imgseq_params* prm, uint8_t* frames, void* stream) {
  if (!img || !prm || !frames) return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: null argument");
  if (mu < 1 || na < 1 || mv < 1) return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: empty image");
  if (na > 65535) return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: at most 65535 frames per call");
  if (prm->n_u < 4 || prm->n_v < 4 || prm->n_u % 4 || prm->n_v % 4)
    return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: frame dimensions must be positive multiples of 4");
  if (prm->n_copies < 1 || prm->n_copies > VAMX_IMGSEQ_MAX_COPIES)
    return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: n_copies out of range");
  if (prm->bit_depth < 1 || prm->bit_depth > 32)
    return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: bit_depth must be in 1..32");
  if (prm->u1 < 0 || (int64_t)prm->u1 + mu > prm->n_u)
    return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: image exceeds the frame in u");
  for (int c = 0; c < prm->n_copies; ++c)
    if (prm->v1[c] < 0 || (int64_t)prm->v1[c] + mv > prm->n_v)
      return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: image copy exceeds the frame in v");
  if ((uintptr_t)frames % 4) return set_error(VAMX_ERR_ARG, "vamx_imgseq_compose: frames must be 4-byte aligned");
  // a NaN normalisation value (a percentile of data holding NaN) makes every
  // sample NaN and every byte 0, as the reference's cast of NaN does
  ComposeDev d;
  d.n_u = prm->n_u;
  d.n_v = prm->n_v;
  d.u1 = prm->u1;
  d.n_copies = prm->n_copies;
  d.bit_depth = prm->bit_depth;
  d.normalize = prm->normalize ? 1 : 0;
  d.flip_u = prm->flip_u ? 1 : 0;
  d.flip_v = prm->flip_v ? 1 : 0;
  d.norm_value = prm->norm_value;
  d.max_value = prm->bit_depth == 32 ? 4294967295.0 : (double)((1ull << prm->bit_depth) - 1ull);
  d.intensity_scale = prm->intensity_scale;
  for (int c = 0; c < VAMX_IMGSEQ_MAX_COPIES; ++c) d.v1[c] = c < prm->n_copies ? prm->v1[c] : 0;
  // every frame byte zeroed once, then the image's tiles into every copy
  hipStream_t s = (hipStream_t)stream;
  const long long nbytes = (long long)na * prm->n_v * prm->n_u;   // a multiple of 16 (n_u, n_v multiples of 4)
  const long long cblocks = std::min<long long>(8192, (nbytes / 16 + 255) / 256);
  if ((uintptr_t)frames % 16 == 0)
    hipLaunchKernelGGL(imgseq_clear<true>, dim3((unsigned)cblocks), dim3(256), 0, s, frames, nbytes);
  else
    hipLaunchKernelGGL(imgseq_clear<false>, dim3((unsigned)cblocks), dim3(256), 0, s, frames, nbytes);
  d.wide = (uintptr_t)frames % 16 == 0 && prm->n_u % 16 == 0;
  d.tile_u0 = prm->u1 / kTile;
  const int tu1 = (prm->u1 + (int)mu - 1) / kTile;
  const dim3 grid(tu1 - d.tile_u0 + 1, (unsigned)((mv + kTile - 1) / kTile), (unsigned)na);
  hipLaunchKernelGGL(imgseq_compose, grid, dim3(256), 0, s, d, img, (long long)mu, (long long)na, (long long)mv,
                     frames);
  VAMX_HIP(hipGetLastError());
  return VAMX_OK;
}
