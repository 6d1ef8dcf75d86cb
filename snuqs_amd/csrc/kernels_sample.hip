// kernels_sample.hip -- sampling from |psi|^2 (simulation.py:217-220).
//
// numpy's RandomState.choice(N, p=p, size=k) returns
// searchsorted(cdf, u, side='right') with cdf = cumsum(p) / cumsum(p)[-1],
// where cumsum is the sequential float64 recurrence c_i = fl(c_{i-1} + p_i)
// and u = random_sample(k).  The sampler takes u from the caller.
//
// Fast mode: cdf by a deterministic FP64 parallel scan (block scans + a scan
// of block totals); it differs from the sequential recurrence by rounding.
//
// Exact mode reproduces the recurrence bit for bit.  While c stays inside one
// binade [2^e, 2^(e+1)) every value is an integer multiple of u = 2^(e-52), so
// fl(c + p) = (C + d) u with d = p/u rounded to nearest; the increments d do
// not depend on c except at exact ties (p/u = k + 1/2, broken towards the even
// result, i.e. by the parity of C).  A run of elements inside one binade is
// therefore a map C -> C + D(parity of C), and such maps compose.
//
// The elements are cut into tiles of 4096.  A fast FP64 scan of the tile sums
// bounds c at each tile's start, which leaves one or two candidate binades; one
// pass forms each tile's map for them.  One workgroup then walks the tiles,
// 1024 maps per scan; where a scan shows that c leaves the binade inside a
// tile, that tile's elements are gone through (the crossing element is added
// with one ordinary double add).  That gives the exact c at every tile's
// start; a last pass writes the cdf inside the tiles that some uniform falls
// into, the last entry of every 16, and a sample adds up the elements of its
// 16.  Nothing waits for the host.  The state is read four times (norm, sums,
// maps, cdf): 2.1 GB at 2^26 complex64 amplitudes, 0.34 ms at copy rate;
// measured 0.98 ms (norm 0.1, sums 0.09, maps 0.13, chain 0.28, a serial chain of
// some 70 scans, cdf 0.16 + 0.06, search 0.02; with the whole cdf written 1.10 ms,
// cdf 0.24 of it), 20 ms with an
// epoch of launches and host reads per binade.  Inputs that are not finite and
// non-negative take the older route, an epoch of launches per binade driven by
// the host.
#include <algorithm>
#include <cmath>
#include <vector>

#include "kernels.hpp"
#include "kernels_reduce.hpp"

namespace sq {

constexpr int kScanItems = 16;
constexpr int kScanTile = kBlock * kScanItems;  // 4096 elements per block

// ---- generic in-place inclusive scan (double or int64) ---------------------
template <typename T>
__device__ void block_scan_tile(T *data, uint64_t n, uint64_t tile, T carry_in,
                                bool use_carry, T *tile_total) {
  __shared__ T s[kScanTile];
  __shared__ T tsum[kBlock];
  const uint64_t base = tile * kScanTile;
  for (int e = threadIdx.x; e < kScanTile; e += kBlock) {
    const uint64_t i = base + e;
    s[e] = i < n ? data[i] : T(0);
  }
  __syncthreads();
  // sequential scan of this thread's run
  T run = 0;
  const int o = threadIdx.x * kScanItems;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    run = (j == 0) ? s[o] : run + s[o + j];
    s[o + j] = run;
  }
  tsum[threadIdx.x] = run;
  __syncthreads();
  // Hillis-Steele inclusive scan of the thread totals
  for (int w = 1; w < kBlock; w <<= 1) {
    T v = (int)threadIdx.x >= w ? tsum[threadIdx.x - w] : T(0);
    __syncthreads();
    if ((int)threadIdx.x >= w) tsum[threadIdx.x] = tsum[threadIdx.x] + v;
    __syncthreads();
  }
  const T excl = threadIdx.x ? tsum[threadIdx.x - 1] : T(0);
  if (tile_total && threadIdx.x == kBlock - 1) *tile_total = tsum[kBlock - 1];
  if (use_carry || threadIdx.x) {
    const T add = use_carry ? (threadIdx.x ? carry_in + excl : carry_in) : excl;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) s[o + j] = s[o + j] + add;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kScanTile; e += kBlock) {
    const uint64_t i = base + e;
    if (i < n) data[i] = s[e];
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_scan_totals(const T *data, uint64_t n, T *totals) {
  // tile totals only (sum of the tile in scan order)
  __shared__ T s[kScanTile];
  __shared__ T tsum[kBlock];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
  for (int e = threadIdx.x; e < kScanTile; e += kBlock) {
    const uint64_t i = base + e;
    s[e] = i < n ? data[i] : T(0);
  }
  __syncthreads();
  T run = 0;
  const int o = threadIdx.x * kScanItems;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) run = (j == 0) ? s[o] : run + s[o + j];
  tsum[threadIdx.x] = run;
  __syncthreads();
  for (int w = 1; w < kBlock; w <<= 1) {
    T v = (int)threadIdx.x >= w ? tsum[threadIdx.x - w] : T(0);
    __syncthreads();
    if ((int)threadIdx.x >= w) tsum[threadIdx.x] = tsum[threadIdx.x] + v;
    __syncthreads();
  }
  if (threadIdx.x == kBlock - 1) totals[blockIdx.x] = tsum[kBlock - 1];
}

template <typename T>
__global__ void __launch_bounds__(kBlock)
    k_scan_apply(T *data, uint64_t n, const T *scanned_totals) {
  const uint64_t tile = blockIdx.x;
  const T carry = tile ? scanned_totals[tile - 1] : T(0);
  block_scan_tile<T>(data, n, tile, carry, tile != 0, nullptr);
}

static uint64_t ntiles(uint64_t n) { return (n + kScanTile - 1) / kScanTile; }

template <typename T>
static size_t scan_scratch(uint64_t n) {
  size_t b = 0;
  while (n > 1) {
    n = ntiles(n);
    b += n * sizeof(T);
    if (n <= 1) break;
  }
  return b + 256;
}

// In-place inclusive scan; scratch holds the per-level tile totals.
template <typename T>
static int scan_inplace(T *data, uint64_t n, T *scratch, hipStream_t st) {
  if (n == 0) return SQ_OK;
  const uint64_t nt = ntiles(n);
  if (nt == 1) {
    hipLaunchKernelGGL(k_scan_apply<T>, dim3(1), dim3(kBlock), 0, st, data, n,
                       (const T *)nullptr);
    SQ_HIP(hipGetLastError());
    return SQ_OK;
  }
  T *totals = scratch;
  hipLaunchKernelGGL(k_scan_totals<T>, dim3((unsigned)nt), dim3(kBlock), 0, st,
                     (const T *)data, n, totals);
  SQ_HIP(hipGetLastError());
  SQ_TRY(scan_inplace<T>(totals, nt, scratch + nt, st));
  hipLaunchKernelGGL(k_scan_apply<T>, dim3((unsigned)nt), dim3(kBlock), 0, st, data,
                     n, (const T *)totals);
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}

// ---- exact-mode epoch kernels ----------------------------------------------
// Increment of p in units of u (ulp of the current binade): d = nearest
// integer, tie flag when p/u is exactly k + 1/2 (d holds k), overflow flag
// when the element alone reaches the top of the binade.
__global__ void __launch_bounds__(kBlock)
    k_increments(const double *__restrict__ p, uint64_t a, uint64_t len,
                 int shift, int64_t *__restrict__ d, int32_t *__restrict__ tie) {
  for (uint64_t m = (uint64_t)blockIdx.x * kBlock + threadIdx.x; m < len;
       m += (uint64_t)gridDim.x * kBlock) {
    const double q = ldexp(p[a + m], shift);  // exact power-of-two scaling
                                              // (inf on overflow, flagged below)
    int64_t di;
    int32_t t = 0;
    if (q >= 9007199254740992.0) {  // 2^53: leaves the binade on its own
      di = (int64_t)1 << 53;
    } else {
      const double k = floor(q);
      const double fr = q - k;  // exact
      di = (int64_t)k;
      if (fr > 0.5) di += 1;
      else if (fr == 0.5) t = 1;
    }
    d[m] = di;
    tie[m] = t;
  }
}

// Resolve ties in order (one thread).  tie holds the inclusive scan of the
// tie flags, d the inclusive scan of the increments; tiepos the positions.
// adj[r] = number of ties among 0..r that rounded up.
__global__ void k_compact_ties(const int32_t *__restrict__ tie_scan, uint64_t len,
                               uint64_t *tiepos) {
  for (uint64_t m = (uint64_t)blockIdx.x * kBlock + threadIdx.x; m < len;
       m += (uint64_t)gridDim.x * kBlock) {
    const int32_t prev = m ? tie_scan[m - 1] : 0;
    if (tie_scan[m] != prev) tiepos[prev] = m;
  }
}

__global__ void k_resolve_ties(const int64_t *__restrict__ dscan,
                               const uint64_t *__restrict__ tiepos, int ntie,
                               int64_t c0, int32_t *adj) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  int32_t up = 0;
  for (int r = 0; r < ntie; ++r) {
    const uint64_t m = tiepos[r];
    // C after element m if the tie rounds down: c0 + dscan[m] + up
    const int64_t down = c0 + dscan[m] + up;
    if (down & 1) ++up;  // halfway between down (odd) and down+1 (even)
    adj[r] = up;
  }
}

// C_m = c0 + dscan[m] + (ties at positions <= m rounded up); first m with
// C_m >= 2^53 is the element that leaves the binade.
__global__ void __launch_bounds__(kBlock)
    k_epoch_values(const int64_t *__restrict__ dscan, uint64_t len, int64_t c0,
                   const uint64_t *__restrict__ tiepos, const int32_t *__restrict__ adj,
                   int ntie, int64_t *__restrict__ cval, unsigned long long *cross) {
  for (uint64_t m = (uint64_t)blockIdx.x * kBlock + threadIdx.x; m < len;
       m += (uint64_t)gridDim.x * kBlock) {
    int lo = 0, hi = ntie;  // number of ties with position <= m
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (tiepos[mid] <= m) lo = mid + 1; else hi = mid;
    }
    const int64_t cm = c0 + dscan[m] + (lo ? adj[lo - 1] : 0);
    cval[m] = cm;
    if (cm >= ((int64_t)1 << 53)) atomicMin(cross, (unsigned long long)m);
  }
}

// cdf[a + m] = C_m * u for m < stop; the crossing element (if any) is added
// with one double add by thread 0 of block 0 afterwards.
__global__ void __launch_bounds__(kBlock)
    k_epoch_write(const int64_t *__restrict__ cval, uint64_t a, uint64_t stop,
                  double u, double *__restrict__ cdf) {
  for (uint64_t m = (uint64_t)blockIdx.x * kBlock + threadIdx.x; m < stop;
       m += (uint64_t)gridDim.x * kBlock)
    cdf[a + m] = (double)cval[m] * u;  // exact: C_m < 2^53
}

__global__ void k_epoch_cross(const double *__restrict__ p, double *cdf, uint64_t pos,
                              double *cval_out) {
  if (threadIdx.x || blockIdx.x) return;
  const double c = (pos == 0) ? p[0] : cdf[pos - 1] + p[pos];
  cdf[pos] = c;
  *cval_out = c;
}

// ---- search ------------------------------------------------------------------
__global__ void __launch_bounds__(kBlock)
    k_search(const double *__restrict__ cdf, uint64_t n, const double *__restrict__ u,
             uint64_t shots, int64_t *__restrict__ out) {
  const double total = cdf[n - 1];
  for (uint64_t s = (uint64_t)blockIdx.x * kBlock + threadIdx.x; s < shots;
       s += (uint64_t)gridDim.x * kBlock) {
    const double v = u[s];
    uint64_t lo = 0, hi = n;
    while (lo < hi) {
      const uint64_t mid = lo + ((hi - lo) >> 1);
      if (cdf[mid] / total <= v) lo = mid + 1; else hi = mid;
    }
    out[s] = (int64_t)lo;
  }
}

int launch_search(const double *cdf, uint64_t n, const double *u_dev, uint64_t shots,
                  int64_t *out_dev, hipStream_t st) {
  if (shots == 0) return SQ_OK;
  hipLaunchKernelGGL(k_search, sweep_grid(shots, kBlock), dim3(kBlock), 0, st, cdf, n, u_dev,
                     shots, out_dev);
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}

// ---- exact mode by tiles -----------------------------------------------------
constexpr int kTileThreads = 1024;
constexpr int kTileItems = 4;
constexpr int kTile = kTileThreads * kTileItems;
// Of a tile's cdf the last entry of every kGroup elements is kept.
constexpr int kGroup = 16;
constexpr int kTileGroups = kTile / kGroup;
constexpr int kGroupThreads = kGroup / kTileItems;
__device__ __forceinline__ bool group_end(int i, int cnt) {
  return (i & (kGroup - 1)) == kGroup - 1 || i == cnt - 1;
}
constexpr double kTop = 9007199254740992.0;  // 2^53: C has left the binade

// What a tile does to C (integers held as doubles: exact below 2^53, and sums
// that reach 2^53 stay there): C -> C + d[C & 1] in binade e, C + d[2 + (C & 1)]
// in binade e + 1 (both only where kHasNext).
struct TileMap {
  double d[4];
  int e;
  int flags;
};
enum { kAllZero = 1, kHasNext = 2, kTies = 4 };

__device__ __forceinline__ bool odd(double x) {
  const double h = x * 0.5;
  return h != floor(h);
}
__device__ __forceinline__ int binade(double c) {
  const int e = (int)((__double_as_longlong(c) >> 52) & 0x7ff) - 1023;
  return e < -1022 ? -1022 : e;  // subnormals share the first binade's ulp
}
// x 2^k, exact unless it leaves the range of doubles (k uniform): one product
// where 2^k is a normal double, and ldexp beyond.
struct Scale {
  double f;
  int k;
  __device__ explicit Scale(int k_)
      : f(k_ >= -1022 && k_ <= 1023 ? __longlong_as_double((int64_t)(k_ + 1023) << 52) : 0.0),
        k(k_) {}
  __device__ __forceinline__ double operator()(double x) const { return f != 0.0 ? x * f : ldexp(x, k); }
};
// Increments of p (in ulps of the binade that `up` scales by) for C even / odd.
__device__ __forceinline__ void increments(double p, const Scale &up, double &d0, double &d1) {
  const double q = up(p);
  const double r = (q + 0x1p52) - 0x1p52;  // nearest integer, ties to even
  d0 = d1 = q < 0x1p52 ? r : q;
  if (fabs(q - d0) == 0.5) {
    const double k = floor(q), o = odd(k) ? 1.0 : 0.0;
    d0 = k + o;
    d1 = k + (1.0 - o);
  }
}
// (a0, a1) followed by (b0, b1).
__device__ __forceinline__ void then(double &a0, double &a1, double b0, double b1) {
  a0 += odd(a0) ? b1 : b0;
  a1 += odd(a1) ? b0 : b1;
}

// Exclusive scan over the workgroup of the maps (d0, d1): on return (d0, d1) is
// the composition of the maps of all lower threads, (t0, t1) that of all.
__device__ __forceinline__ void scan_maps(double &d0, double &d1, double &t0, double &t1) {
  constexpr int W = kTileThreads / 64;
  __shared__ double w0[W], w1[W];
  __shared__ int wp[W];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool wpairs = __any(d0 != d1);
  double i0 = d0, i1 = d1;
  if (!wpairs) {  // no ties in this wave: plain sums
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double p0 = __shfl_up(i0, o);
      if (lane >= o) i0 += p0;
    }
    i1 = i0;
  } else {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      double p0 = __shfl_up(i0, o), p1 = __shfl_up(i1, o);
      if (lane >= o) {
        then(p0, p1, i0, i1);
        i0 = p0;
        i1 = p1;
      }
    }
  }
  double e0 = __shfl_up(i0, 1), e1 = wpairs ? __shfl_up(i1, 1) : e0;
  if (lane == 0) e0 = e1 = 0.0;
  __syncthreads();  // an earlier call's reads are done
  if (lane == 63) {
    w0[wave] = i0;
    w1[wave] = i1;
    wp[wave] = wpairs;
  }
  __syncthreads();
  int pairs = 0;
#pragma unroll
  for (int v = 0; v < W; ++v) pairs |= wp[v];
  double a0 = 0.0, a1 = 0.0, s0 = 0.0, s1 = 0.0;
  if (!pairs) {
#pragma unroll
    for (int v = 0; v < W; ++v) {
      if (v == wave) s0 = a0;
      a0 += w0[v];
    }
    t0 = t1 = a0;
    d0 = d1 = s0 + e0;
    return;
  }
  for (int v = 0; v < W; ++v) {
    if (v == wave) {
      s0 = a0;
      s1 = a1;
    }
    then(a0, a1, w0[v], w1[v]);
  }
  t0 = a0;
  t1 = a1;
  then(s0, s1, e0, e1);
  d0 = s0;
  d1 = s1;
}

// Smallest of the threads' values.
__device__ __forceinline__ int block_min(int v) {
  __shared__ int m[kTileThreads / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) m[threadIdx.x >> 6] = v;
  __syncthreads();
  int r = m[0];
#pragma unroll
  for (int w = 1; w < kTileThreads / 64; ++w) r = min(r, m[w]);
  return r;
}

// The recurrence over one tile's elements (thread t holds items 4t .. 4t + 3,
// cnt in all) from c; writes the groups' last cdf entries to out and returns c
// after the tile.  Every round of the loop ends the tile or passes one
// element that starts a binade.
__device__ __forceinline__ double walk_tile(const double (&x)[kTileItems], int cnt, double c,
                                            double *__restrict__ out) {
  __shared__ double sc;
  const int i0 = threadIdx.x * kTileItems;
  int s = 0;  // elements before s are done
  while (s < cnt) {
    double v[kTileItems], start = 0.0;  // C (0 while c is 0) after each item
    int f = kTile, first = kTile;
    const int e = binade(c);
    const Scale down(e - 52);
    if (c == 0.0) {
#pragma unroll
      for (int j = kTileItems - 1; j >= 0; --j) {
        v[j] = 0.0;
        if (i0 + j >= s && i0 + j < cnt && x[j] > 0.0) f = i0 + j;
      }
      first = block_min(f);
    } else {
      if (!(c > 0.0 && c < __builtin_inf())) return c;  // not a probability: given up
      const Scale up(52 - e);
      const double C0 = up(c);
      double d0[kTileItems], d1[kTileItems];
      double t0 = 0.0, t1 = 0.0, a0, a1;
      bool pairs = false;
#pragma unroll
      for (int j = 0; j < kTileItems; ++j) {
        d0[j] = d1[j] = 0.0;
        if (i0 + j >= s && i0 + j < cnt) increments(x[j], up, d0[j], d1[j]);
        pairs |= d0[j] != d1[j];
      }
      if (!pairs) {
        t0 = t1 = d0[0] + d0[1] + d0[2] + d0[3];
      } else {
#pragma unroll
        for (int j = 0; j < kTileItems; ++j) then(t0, t1, d0[j], d1[j]);
      }
      scan_maps(t0, t1, a0, a1);
      const bool o = odd(C0);
      start = C0 + (o ? t1 : t0);
      double C = start;
#pragma unroll
      for (int j = 0; j < kTileItems; ++j) {
        C += pairs && odd(C) ? d1[j] : d0[j];
        v[j] = C;
      }
      if (C0 + (o ? a1 : a0) >= kTop) {  // leaves the binade in this tile
#pragma unroll
        for (int j = kTileItems - 1; j >= 0; --j)
          if (v[j] >= kTop) f = i0 + j;
        first = block_min(f);
      }
    }
#pragma unroll
    for (int j = 0; j < kTileItems; ++j)
      if (i0 + j >= s && i0 + j < first && group_end(i0 + j, cnt) && i0 + j < cnt)
        out[(i0 + j) / kGroup] = down(v[j]);
    const bool last = first >= cnt;  // stays in the binade to the tile's end
    if (last ? (int)threadIdx.x == (cnt - 1) / kTileItems : f == first) {
      double l = start, px = 0.0;  // C before (after, at the end) the element
#pragma unroll
      for (int j = kTileItems - 1; j >= 0; --j) {
        if (last) {
          if (i0 + j == cnt - 1) l = v[j];
        } else if (i0 + j == first) {
          px = x[j];
          if (j) l = v[j - 1];
        }
      }
      sc = down(l) + px;
      if (!last && group_end(first, cnt)) out[first / kGroup] = sc;
    }
    __syncthreads();
    c = sc;
    __syncthreads();
    s = first + 1;
  }
  return c;
}

// Where the probabilities come from: an array, or |a|^2 of a state's amplitudes
// in FP64 without contraction, divided by *norm2 unless that is null (the
// values of k_probabilities and k_probabilities_div).
struct FromArray {
  const double *p;
  __device__ __forceinline__ double one(uint64_t i) const { return p[i]; }
  __device__ __forceinline__ void four(uint64_t i, double (&x)[kTileItems]) const {
    if (((uintptr_t)p & 15) == 0) {
      const double2 a = *reinterpret_cast<const double2 *>(p + i);
      const double2 b = *reinterpret_cast<const double2 *>(p + i + 2);
      x[0] = a.x;
      x[1] = a.y;
      x[2] = b.x;
      x[3] = b.y;
    } else {
#pragma unroll
      for (int j = 0; j < kTileItems; ++j) x[j] = p[i + j];
    }
  }
};
template <typename T>
struct FromState {
  const T *sv;
  const double *norm2;
  __device__ __forceinline__ double prob(double re, double im) const {
#pragma clang fp contract(off)
    const double q = re * re + im * im;
    return norm2 ? q / *norm2 : q;
  }
  __device__ __forceinline__ double one(uint64_t i) const { return prob(sv[i].x, sv[i].y); }
  __device__ __forceinline__ void four(uint64_t i, double (&x)[kTileItems]) const {
    T a[kTileItems];
    if (sizeof(T) == 8 && ((uintptr_t)sv & 15) == 0) {
      const float4 *q = reinterpret_cast<const float4 *>(sv + i);
      const float4 u = q[0], v = q[1];
      a[0].x = u.x, a[0].y = u.y, a[1].x = u.z, a[1].y = u.w;
      a[2].x = v.x, a[2].y = v.y, a[3].x = v.z, a[3].y = v.w;
    } else {
#pragma unroll
      for (int j = 0; j < kTileItems; ++j) a[j] = sv[i + j];
    }
#pragma unroll
    for (int j = 0; j < kTileItems; ++j) x[j] = prob(a[j].x, a[j].y);
  }
};

// This thread's items of a tile and the tile's element count.
template <typename S>
__device__ __forceinline__ int load_tile(const S &src, uint64_t n, uint64_t tile,
                                         double (&x)[kTileItems]) {
  const uint64_t base = tile * kTile;
  const int cnt = (int)(n - base < (uint64_t)kTile ? n - base : (uint64_t)kTile);
  const int i0 = threadIdx.x * kTileItems;
  if (cnt == kTile) {
    src.four(base + i0, x);
  } else {
#pragma unroll
    for (int j = 0; j < kTileItems; ++j) x[j] = i0 + j < cnt ? src.one(base + i0 + j) : 0.0;
  }
  return cnt;
}

// The tile of this workgroup: a launch over nt tiles (a power of two) is
// tile_grid(nt), in two dimensions where one would hold 2^32 work-items (2^34
// elements).
constexpr uint64_t kTileGridX = 1ull << 20;
static dim3 tile_grid(uint64_t nt) {
  const uint64_t x = std::min(nt, kTileGridX);
  return dim3((unsigned)x, (unsigned)((nt + x - 1) / x));
}
__device__ __forceinline__ uint64_t tile_index() {
  return (uint64_t)blockIdx.y * gridDim.x + blockIdx.x;
}

// Sum of each tile (any order: it only bounds c); *bad is set by an element
// that is negative or not finite.
template <typename S>
__global__ void __launch_bounds__(kTileThreads)
    k_tile_sums(S src, uint64_t n, double *__restrict__ sums, int *__restrict__ bad) {
  __shared__ double w[kTileThreads / 64];
  const uint64_t tile = tile_index();
  double x[kTileItems];
  load_tile(src, n, tile, x);
  double s = 0.0;
  bool b = false;
#pragma unroll
  for (int j = 0; j < kTileItems; ++j) {
    b |= !(x[j] >= 0.0 && x[j] < __builtin_inf());
    s += x[j];
  }
  if (b) *bad = 1;
  s = wave_sum_d(s);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    s = 0.0;
    for (int v = 0; v < kTileThreads / 64; ++v) s += w[v];
    sums[tile] = s;
  }
}

// Each tile's map for the binades that c may be in at its start: the scanned
// sums' error and the recurrence's own are each below (n + 16) 2^-53 of c.
template <typename S>
__global__ void __launch_bounds__(kTileThreads, 8)
    k_tile_maps(S src, uint64_t n, const double *__restrict__ scanned, TileMap *__restrict__ maps) {
  constexpr int W = kTileThreads / 64;
  __shared__ double w[2][W];
  __shared__ int wf[W];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t tile = tile_index();
  double x[kTileItems];
  load_tile(src, n, tile, x);
  const double a = tile ? scanned[tile - 1] : 0.0;
  const double slack = (double)(n + 16) * 0x1p-51;
  TileMap m{};
  m.e = binade(a * (1.0 - slack));
  if (binade(a * (1.0 + slack)) != m.e) m.flags = kHasNext;
  // increments in both binades (the second is rarely needed), without regard
  // to ties; f bit 0: an element is not zero, bit 1: a tie
  const Scale up0(52 - m.e), up1(51 - m.e);
  double t0 = 0.0, t1 = 0.0;
  int f = 0;
#pragma unroll
  for (int j = 0; j < kTileItems; ++j) {
    double d0, d1;
    increments(x[j], up0, d0, d1);
    f |= (x[j] != 0.0) | (d0 != d1 ? 2 : 0);
    t0 += d0;
    if (m.flags) {
      increments(x[j], up1, d0, d1);
      f |= d0 != d1 ? 2 : 0;
      t1 += d0;
    }
  }
  t0 = wave_sum_d(t0);
  if (m.flags) t1 = wave_sum_d(t1);
  f = (__any(f & 1) ? 1 : 0) | (__any(f & 2) ? 2 : 0);
  if (lane == 0) {
    w[0][wave] = t0;
    w[1][wave] = t1;
    wf[wave] = f;
  }
  __syncthreads();
  f = 0;
  t0 = t1 = 0.0;
#pragma unroll
  for (int v = 0; v < W; ++v) {
    f |= wf[v];
    t0 += w[0][v];
    t1 += w[1][v];
  }
  m.d[0] = m.d[1] = t0;
  m.d[2] = m.d[3] = t1;
  if (!(f & 1)) m.flags |= kAllZero;
  if (f & 2) m.flags |= kTies;
  if (threadIdx.x == 0) maps[tile] = m;
}

// The maps of the tiles that hold ties, which depend on the parity of C.
template <typename S>
__global__ void __launch_bounds__(kTileThreads)
    k_tile_tie_maps(S src, uint64_t n, TileMap *__restrict__ maps) {
  const uint64_t tile = tile_index();
  const int flags = maps[tile].flags, e = maps[tile].e;
  if (!(flags & kTies)) return;
  double x[kTileItems];
  load_tile(src, n, tile, x);
  for (int k = 0; k < ((flags & kHasNext) ? 2 : 1); ++k) {
    const Scale up(52 - e - k);
    double d0, d1, s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int j = 0; j < kTileItems; ++j) {
      increments(x[j], up, d0, d1);
      then(s0, s1, d0, d1);
    }
    scan_maps(s0, s1, d0, d1);
    if (threadIdx.x == 0) {
      maps[tile].d[2 * k] = d0;
      maps[tile].d[2 * k + 1] = d1;
    }
  }
}

// One workgroup: the exact c before every tile, tile_in[t], and after the
// last, tile_in[nt]; the group ends of the tiles it goes through.
template <typename S>
__global__ void __launch_bounds__(kTileThreads)
    k_tile_chain(S src, uint64_t n, uint64_t nt, const TileMap *__restrict__ maps,
                 double *__restrict__ tile_in, double *__restrict__ ends, int *bad) {
  if (*bad) return;
  __shared__ double sc;
  const int tid = threadIdx.x;
  double c = 0.0;
  TileMap m{}, next{};
  if ((uint64_t)tid < nt) next = maps[tid];
  for (uint64_t t0 = 0; t0 < nt; t0 += kTileThreads) {
    const uint64_t t = t0 + tid;
    m = next;
    if (t + kTileThreads < nt) next = maps[t + kTileThreads];
    for (int s = 0; s < kTileThreads;) {  // tiles before t0 + s are done
      double d0 = 0.0, d1 = 0.0;
      const int e = binade(c);
      const Scale up(52 - e), down(e - 52);
      const double C0 = up(c);
      if (t < nt && tid >= s && !(m.flags & kAllZero)) {
        if (c > 0.0 && e == m.e) {
          d0 = m.d[0];
          d1 = m.d[1];
        } else if (c > 0.0 && (m.flags & kHasNext) && e == m.e + 1) {
          d0 = m.d[2];
          d1 = m.d[3];
        } else {
          d0 = d1 = kTop;  // no map for this binade: gone through below
        }
      }
      double s0 = d0, s1 = d1, a0, a1;
      scan_maps(s0, s1, a0, a1);
      const bool o = odd(C0);
      const double start = C0 + (o ? s1 : s0);
      const double all = C0 + (o ? a1 : a0);
      if (all < kTop) {
        if (t < nt && tid >= s) tile_in[t] = down(start);
        c = down(all);
        break;
      }
      const double end = start + (odd(start) ? d1 : d0);
      const int f = block_min(tid >= s && end >= kTop ? tid : kTileThreads);
      if (t < nt && tid >= s && tid <= f) tile_in[t] = down(start);
      if (tid == f) sc = down(start);
      __syncthreads();
      c = sc;
      double x[kTileItems];
      const int cnt = load_tile(src, n, t0 + f, x);
      c = walk_tile(x, cnt, c, ends + (t0 + f) * kTileGroups);
      if (!(c < __builtin_inf())) {  // the sum overflows (c is uniform): no binade to go on in
        if (tid == 0) *bad = 1;
        return;
      }
      s = f + 1;  // s <= f: every round passes a tile
    }
  }
  if (tid == 0) tile_in[nt] = c;
}

// The tile of each uniform: the first whose end is above it (the entries
// before a tile's end are searched by k_tile_search), marked as needed.
__global__ void __launch_bounds__(kBlock)
    k_tile_find(const double *__restrict__ tile_in, uint64_t nt, const double *__restrict__ u,
                uint64_t shots, int64_t *__restrict__ out, int *__restrict__ need,
                const int *__restrict__ bad) {
  if (*bad) return;
  const double total = tile_in[nt];
  for (uint64_t s = (uint64_t)blockIdx.x * kBlock + threadIdx.x; s < shots;
       s += (uint64_t)gridDim.x * kBlock) {
    const double v = u[s];
    uint64_t lo = 0, hi = nt;
    while (lo < hi) {
      const uint64_t mid = lo + ((hi - lo) >> 1);
      if (tile_in[mid + 1] / total <= v) lo = mid + 1; else hi = mid;
    }
    out[s] = (int64_t)lo;
    if (lo < nt) need[lo] = 1;
  }
}

// How a needed tile gets its group ends: by one plain scan, by a scan with ties, or not
// here (c leaves its binade there: k_tile_chain has written it).
enum class TileCdf { kDone, kPlain, kTied };
__device__ __forceinline__ TileCdf tile_cdf(const double *tile_in, const TileMap *maps, uint64_t t) {
  const double c = tile_in[t];
  if (!(c > 0.0) || binade(c) != binade(tile_in[t + 1]))
    return c == 0.0 && tile_in[t + 1] == 0.0 ? TileCdf::kTied : TileCdf::kDone;
  return maps[t].flags & kTies ? TileCdf::kTied : TileCdf::kPlain;
}

// The group ends of the needed tiles: the plain ones (few registers, so two
// workgroups share a CU) and the others.  Bound by the read of the state; the
// whole cdf, 8 bytes an element, was as much to write as complex64 is to read.
template <typename S>
__global__ void __launch_bounds__(kTileThreads, 8)
    k_tile_cdf(S src, uint64_t n, const double *__restrict__ tile_in,
               const TileMap *__restrict__ maps, const int *__restrict__ need,
               double *__restrict__ ends, const int *__restrict__ bad) {
  constexpr int W = kTileThreads / 64;
  __shared__ double w[W];
  const uint64_t tile = tile_index();
  if (*bad || !need[tile] || tile_cdf(tile_in, maps, tile) != TileCdf::kPlain) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double x[kTileItems];
  load_tile(src, n, tile, x);
  const double c = tile_in[tile];
  const int e = binade(c);
  const Scale up(52 - e), down(e - 52);
  double d1;
#pragma unroll
  for (int j = 0; j < kTileItems; ++j) {
    increments(x[j], up, x[j], d1);
    if (j) x[j] += x[j - 1];
  }
  double i = x[kTileItems - 1];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double p = __shfl_up(i, o);
    if (lane >= o) i += p;
  }
  if (lane == 63) w[wave] = i;
  __syncthreads();
  double start = up(c) + (i - x[kTileItems - 1]);
#pragma unroll
  for (int v = 0; v < W; ++v)
    if (v < wave) start += w[v];
  // (elements past the state's end add nothing)
  if (threadIdx.x % kGroupThreads == kGroupThreads - 1)
    ends[tile * kTileGroups + threadIdx.x / kGroupThreads] =
        down(start + x[kTileItems - 1]);
}

template <typename S>
__global__ void __launch_bounds__(kTileThreads)
    k_tile_cdf_walk(S src, uint64_t n, uint64_t nt, const double *__restrict__ tile_in,
                    const TileMap *__restrict__ maps, const int *__restrict__ need,
                    double *__restrict__ ends, const int *__restrict__ bad) {
  if (*bad) return;
  for (uint64_t t = blockIdx.x; t < nt; t += gridDim.x) {
    if (!need[t] || tile_cdf(tile_in, maps, t) != TileCdf::kTied) continue;
    double x[kTileItems];
    const int cnt = load_tile(src, n, t, x);
    walk_tile(x, cnt, tile_in[t], ends + t * kTileGroups);
  }
}

// out[s]: the uniform's tile on entry, its element on return: the first group
// whose end is above the uniform, then the recurrence itself over its elements.
template <typename S>
__global__ void __launch_bounds__(kBlock)
    k_tile_search(S src, const double *__restrict__ ends, uint64_t n,
                  const double *__restrict__ tile_in, uint64_t nt, const double *__restrict__ u,
                  uint64_t shots, int64_t *__restrict__ out, const int *__restrict__ bad) {
  if (*bad) return;
  const double total = tile_in[nt];
  for (uint64_t s = (uint64_t)blockIdx.x * kBlock + threadIdx.x; s < shots;
       s += (uint64_t)gridDim.x * kBlock) {
    const uint64_t tile = (uint64_t)out[s];
    uint64_t i = n;
    if (tile < nt) {
      const double v = u[s];
      const uint64_t left = n - tile * kTile;
      const int ngroups = left < kTile ? ((int)left + kGroup - 1) / kGroup : kTileGroups;
      const double *end = ends + tile * kTileGroups;
      int lo = 0, hi = ngroups - 1;  // the tile's end is above v
      while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (end[mid] / total <= v) lo = mid + 1; else hi = mid;
      }
      double c = lo ? end[lo - 1] : tile_in[tile];
      i = tile * kTile + (uint64_t)lo * kGroup;
      const int cnt = (int)(n - i < (uint64_t)kGroup ? n - i : (uint64_t)kGroup);
      double x[kGroupThreads][kTileItems];
#pragma unroll
      for (int q = 0; q < kGroupThreads; ++q) {
        if (cnt == kGroup) {
          src.four(i + q * kTileItems, x[q]);
        } else {
#pragma unroll
          for (int j = 0; j < kTileItems; ++j)
            x[q][j] = q * kTileItems + j < cnt ? src.one(i + q * kTileItems + j) : 0.0;
        }
      }
      int below = 0;  // elements whose cdf is not above v (the cdf never falls)
#pragma unroll
      for (int j = 0; j < kGroup; ++j) {
        c += x[j / kTileItems][j % kTileItems];
        below += j < cnt - 1 && c / total <= v;
      }
      i += below;
    }
    out[s] = (int64_t)i;
  }
}

static uint64_t tile_count(uint64_t n) { return (n + kTile - 1) / kTile; }

size_t sample_exact_scratch_bytes(uint64_t n) {
  const uint64_t nt = tile_count(n);
  return nt * ((1 + kTileGroups) * sizeof(double) + sizeof(TileMap) + sizeof(int)) +
         (nt + 1) * sizeof(double) + scan_scratch<double>(nt) + 8 * 256;
}

// ---- host driver -----------------------------------------------------------
size_t sample_scratch_bytes(uint64_t n, bool exact) {
  size_t b = scan_scratch<double>(n) + 4096;
  if (exact) {
    // increments + tie flags + scanned values for one epoch segment (<= n),
    // tie positions and adjustments, scan scratch for int64 and int32
    b += n * (sizeof(int64_t) * 2 + sizeof(int32_t)) + scan_scratch<int64_t>(n) +
         scan_scratch<int32_t>(n) + 4096;
  }
  return b;
}

static inline char *align_up(char *p) {
  return (char *)(((uintptr_t)p + 255) & ~(uintptr_t)255);
}

template <typename S>
static int sample_exact_t(const S &src, uint64_t n, const double *u_dev,
                          uint64_t shots, int64_t *out_dev, void *scratch, const int **bad_dev,
                          hipStream_t st) {
  const uint64_t nt = tile_count(n);
  char *w = align_up((char *)scratch);
  int *need = (int *)w;  // nt flags, then *bad
  w = align_up(w + (nt + 1) * sizeof(int));
  double *sums = (double *)w;
  w = align_up(w + nt * sizeof(double));
  double *tile_in = (double *)w;
  w = align_up(w + (nt + 1) * sizeof(double));
  TileMap *maps = (TileMap *)w;
  w = align_up(w + nt * sizeof(TileMap));
  double *ends = (double *)w;
  w = align_up(w + nt * kTileGroups * sizeof(double));
  int *bad = need + nt;
  SQ_HIP(hipMemsetAsync(need, 0, (nt + 1) * sizeof(int), st));
  const dim3 g = tile_grid(nt), b(kTileThreads);
  hipLaunchKernelGGL(k_tile_sums<S>, g, b, 0, st, src, n, sums, bad);
  SQ_HIP(hipGetLastError());
  SQ_TRY(scan_inplace<double>(sums, nt, (double *)w, st));
  hipLaunchKernelGGL(k_tile_maps<S>, g, b, 0, st, src, n, (const double *)sums, maps);
  hipLaunchKernelGGL(k_tile_tie_maps<S>, g, b, 0, st, src, n, maps);
  hipLaunchKernelGGL(k_tile_chain<S>, dim3(1), b, 0, st, src, n, nt, (const TileMap *)maps,
                     tile_in, ends, bad);
  hipLaunchKernelGGL(k_tile_find, sweep_grid(shots, kBlock), dim3(kBlock), 0, st,
                     (const double *)tile_in, nt, u_dev, shots, out_dev, need, (const int *)bad);
  hipLaunchKernelGGL(k_tile_cdf<S>, g, b, 0, st, src, n, (const double *)tile_in,
                     (const TileMap *)maps, (const int *)need, ends, (const int *)bad);
  hipLaunchKernelGGL(k_tile_cdf_walk<S>, dim3((unsigned)std::min<uint64_t>(nt, 1024)), b, 0, st,
                     src, n, nt, (const double *)tile_in, (const TileMap *)maps,
                     (const int *)need, ends, (const int *)bad);
  hipLaunchKernelGGL(k_tile_search<S>, sweep_grid(shots, kBlock), dim3(kBlock), 0, st, src,
                     (const double *)ends, n, (const double *)tile_in, nt, u_dev, shots, out_dev,
                     (const int *)bad);
  SQ_HIP(hipGetLastError());
  *bad_dev = bad;
  return SQ_OK;
}

int sample_exact(const double *p, uint64_t n, const double *u_dev, uint64_t shots,
                 int64_t *out_dev, void *scratch, const int **bad_dev, hipStream_t st) {
  return sample_exact_t(FromArray{p}, n, u_dev, shots, out_dev, scratch, bad_dev, st);
}

int sample_exact_state(const void *sv, sq_dtype_t dt, const double *norm2_dev, uint64_t n,
                       const double *u_dev, uint64_t shots, int64_t *out_dev,
                       void *scratch, const int **bad_dev, hipStream_t st) {
  if (dt == SQ_COMPLEX64)
    return sample_exact_t(FromState<float2>{(const float2 *)sv, norm2_dev}, n, u_dev, shots,
                          out_dev, scratch, bad_dev, st);
  return sample_exact_t(FromState<double2>{(const double2 *)sv, norm2_dev}, n, u_dev, shots,
                        out_dev, scratch, bad_dev, st);
}

int sample_cdf(const double *p, uint64_t n, double *cdf, bool exact, void *scratch,
               size_t scratch_bytes, hipStream_t st) {
  if (scratch_bytes < sample_scratch_bytes(n, exact))
    return fail(SQ_ERR_INVALID, "internal: sampler scratch too small");
  char *w = align_up((char *)scratch);
  double *dscr = (double *)w;
  w = align_up(w + scan_scratch<double>(n));
  SQ_HIP(hipMemcpyAsync(cdf, p, n * sizeof(double), hipMemcpyDeviceToDevice, st));
  SQ_TRY(scan_inplace<double>(cdf, n, dscr, st));  // fast cdf (c')
  if (!exact) return SQ_OK;

  // Exact mode.  The fast cdf c' bounds the position where each binade ends:
  // |c_m - c'_m| <= (m + 1) * 2^-52 * c'_m covers the rounding of both sums.
  int64_t *dinc = (int64_t *)w;
  w = align_up(w + n * sizeof(int64_t));
  int64_t *cval = (int64_t *)w;
  w = align_up(w + n * sizeof(int64_t));
  int32_t *tie = (int32_t *)w;
  w = align_up(w + n * sizeof(int32_t));
  int64_t *iscr = (int64_t *)w;
  w = align_up(w + scan_scratch<int64_t>(n));
  int32_t *tscr = (int32_t *)w;
  w = align_up(w + scan_scratch<int32_t>(n));

  // Host copies of c' are read by binary search through small D2H reads.
  auto read_d = [&](const double *src, double *dst) -> int {
    SQ_HIP(hipMemcpyAsync(dst, src, sizeof(double), hipMemcpyDeviceToHost, st));
    SQ_HIP(hipStreamSynchronize(st));
    return SQ_OK;
  };
  // first index m >= lo with c'_m > thr (n if none); c' is non-decreasing.
  auto first_above = [&](uint64_t lo, double thr, uint64_t *res) -> int {
    uint64_t a = lo, b = n;
    double v;
    while (a < b) {
      const uint64_t mid = a + (b - a) / 2;
      SQ_TRY(read_d(cdf + mid, &v));
      if (v > thr) b = mid; else a = mid + 1;
    }
    *res = a;
    return SQ_OK;
  };

  // Leading zeros: c_m = 0 exactly until the first positive p (c' is 0 there
  // too), then c = p exactly.
  uint64_t pos;
  SQ_TRY(first_above(0, 0.0, &pos));
  if (pos >= n) return SQ_OK;  // all zero: cdf is all zero as in numpy
  double c;
  {
    // cdf[pos] = 0 + p[pos] = p[pos]
    SQ_HIP(hipMemcpyAsync(cdf + pos, p + pos, sizeof(double), hipMemcpyDeviceToDevice, st));
    SQ_TRY(read_d(p + pos, &c));
  }
  double *dev_c = dscr;  // one double of scratch for the crossing value
  unsigned long long *dev_cross = (unsigned long long *)(dscr + 1);

  while (pos + 1 < n) {
    if (!(c > 0.0) || !std::isfinite(c))
      return fail(SQ_ERR_INVALID, "probabilities must be finite and non-negative");
    int e = std::ilogb(c);
    if (e < -1022) e = -1022;
    const double u = std::ldexp(1.0, e - 52);
    const double top = std::ldexp(1.0, e + 1);
    const int64_t c0 = (int64_t)(c / u);  // exact
    // segment [a, hi): a = pos + 1; hi bounds the crossing from above
    const uint64_t a = pos + 1;
    uint64_t hi;
    {
      const double slack = (double)(n + 1) * std::ldexp(1.0, -52) * 2.0;
      SQ_TRY(first_above(a, top * (1.0 + slack), &hi));
      hi = std::min<uint64_t>(n, hi + 1);
      if (hi <= a) hi = std::min<uint64_t>(n, a + 1);
    }
    const uint64_t len = hi - a;
    const dim3 g = sweep_grid(len, kBlock);
    hipLaunchKernelGGL(k_increments, g, dim3(kBlock), 0, st, p, a, len,
                       52 - e, dinc, tie);
    SQ_HIP(hipGetLastError());
    SQ_TRY(scan_inplace<int64_t>(dinc, len, iscr, st));
    SQ_TRY(scan_inplace<int32_t>(tie, len, tscr, st));
    int32_t ntie = 0;
    SQ_HIP(hipMemcpyAsync(&ntie, tie + len - 1, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    SQ_HIP(hipStreamSynchronize(st));
    // tie positions and adjustments live in the (now free) scan scratch
    uint64_t *tpos = (uint64_t *)iscr;
    int32_t *adj = (int32_t *)tscr;
    if ((size_t)ntie * sizeof(uint64_t) > scan_scratch<int64_t>(n) ||
        (size_t)ntie * sizeof(int32_t) > scan_scratch<int32_t>(n))
      return fail(SQ_ERR_UNSUPPORTED, "exact sampler: too many rounding ties");
    if (ntie > 0) {
      hipLaunchKernelGGL(k_compact_ties, g, dim3(kBlock), 0, st,
                         (const int32_t *)tie, len, tpos);
      hipLaunchKernelGGL(k_resolve_ties, dim3(1), dim3(64), 0, st,
                         (const int64_t *)dinc, (const uint64_t *)tpos, (int)ntie, c0, adj);
      SQ_HIP(hipGetLastError());
    }
    const unsigned long long none = ~0ull;
    SQ_HIP(hipMemcpyAsync(dev_cross, &none, sizeof(none), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_epoch_values, g, dim3(kBlock), 0, st, (const int64_t *)dinc,
                       len, c0, (const uint64_t *)tpos, (const int32_t *)adj, (int)ntie,
                       cval, dev_cross);
    SQ_HIP(hipGetLastError());
    unsigned long long cross = 0;
    SQ_HIP(hipMemcpyAsync(&cross, dev_cross, sizeof(cross), hipMemcpyDeviceToHost, st));
    SQ_HIP(hipStreamSynchronize(st));
    const uint64_t stop = (cross == none) ? len : (uint64_t)cross;
    if (stop > 0) {
      hipLaunchKernelGGL(k_epoch_write, sweep_grid(stop, kBlock), dim3(kBlock), 0, st,
                         (const int64_t *)cval, a, stop, u, cdf);
      SQ_HIP(hipGetLastError());
    }
    if (cross == none) {
      if (hi >= n) break;  // reached the end inside this binade
      return fail(SQ_ERR_INVALID,
                  "exact sampler: binade bound violated (probabilities not finite?)");
    }
    pos = a + stop;
    hipLaunchKernelGGL(k_epoch_cross, dim3(1), dim3(64), 0, st, p, cdf, pos, dev_c);
    SQ_HIP(hipGetLastError());
    SQ_TRY(read_d(dev_c, &c));
  }
  return SQ_OK;
}

}  // namespace sq
