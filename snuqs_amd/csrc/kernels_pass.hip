// kernels_pass.hip -- several gates of a program in one sweep over the state.
//
// A workgroup owns a chunk of 2^CB amplitudes (the pass's local bits), moves it
// into LDS, multiplies every block matrix of the pass onto it on the matrix
// cores and writes it back, so a pass reads and writes the state once whatever
// its number of gates.  Blocks act on 4 or 5 of the chunk's bits; a wave takes
// tiles of 32 (complex64) / 16 (complex128) groups, reads a tile's operands
// from LDS, multiplies and writes the tile back in place, with a workgroup
// barrier between blocks.  The LDS slot of chunk index e is linear over GF(2)
// in e's bits (pass_plan.cpp), so an address is a per-lane constant XOR a
// uniform term.
//
// Bound: a 5-target block takes 1.3 ms of FP32 MFMA at 2^30 complex64
// amplitudes and the sweep 2.7 ms of HBM time at copy rate, so one block hides
// under the sweep and from the second on the matrix cores share the time.
// Measured at 2^30 complex64, local bits of four shapes: 0 blocks 3.1-3.9 ms,
// 1 block 3.2-4.3, 2 blocks 4.5-5.8, 3 blocks 5.9-6.6, 4 blocks 7.3-7.7, where
// one block per launch takes 3.1 ms each.  Layered 30-qubit circuit of depth
// 10 in 50 blocks: 155 -> 110 ms; 25-qubit mixed circuit of 175 gates unfused:
// 12.4 -> 1.6 ms.  A loop over several chunks per workgroup with the next
// chunk's loads issued ahead of the products (4 waves, 2 tiles each) measured
// 5-10% slower than one chunk per workgroup: the two workgroups of a CU
// already overlap one's loads with the other's products.
#include <algorithm>

#include "kernels.hpp"
#include "pass_plan.hpp"

namespace sq {

// Workgroups of a pass: one chunk each (a dispatch holds fewer than 2^32
// work-items).
constexpr uint64_t kPassGrid = 1ull << 22;

typedef float pfloatx16 __attribute__((ext_vector_type(16)));
typedef double pdoublex4 __attribute__((ext_vector_type(4)));

// Slot weights of pass_plan.cpp.
template <typename R>
__device__ constexpr uint32_t pass_slot(int i) {
  constexpr uint32_t h64[13] = {1, 2, 4, 8, 16, 15, 23, 14, 5, 25, 6, 19, 26};
  constexpr uint32_t h128[12] = {1, 2, 4, 8, 3, 9, 14, 7, 6, 12, 13, 11};
  if (sizeof(R) == 4) return (i < 5 ? 0u : 1u << i) | h64[i];
  return (i < 4 ? 0u : 1u << i) | h128[i < 12 ? i : 0];
}

// XOR of the weights w[i] whose bit of v is set (v a compile-time constant
// after unrolling, w uniform).
template <int N>
__device__ __forceinline__ uint32_t xor_bits(const uint16_t *w, int v) {
  uint32_t r = 0;
#pragma unroll
  for (int i = 0; i < N; ++i)
    if ((v >> i) & 1) r ^= w[i];
  return r;
}

// XOR of the weights by the bits of a per-lane value.
template <int N>
__device__ __forceinline__ uint32_t xor_lane(const uint16_t *w, uint32_t v) {
  uint32_t r = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) r ^= ((v >> i) & 1) ? (uint32_t)w[i] : 0u;
  return r;
}

// One 5-target block on this wave's tile (complex64): three real products per
// complex one, operands as in k_mfma5_c64.
__device__ __forceinline__ void pass_block5(char *X, const float4 *As, const PassBlock &b, int lane,
                                            uint32_t lb) {
  const int col = lane & 31, half = lane >> 5;
  const uint32_t rd = lb ^ (half ? b.row[0] : 0u), wr = lb ^ (half ? b.row[2] : 0u);
  float2 x[16];
#pragma unroll
  for (int s = 0; s < 16; ++s)
    x[s] = *reinterpret_cast<const float2 *>(X + (rd ^ xor_bits<4>(b.row + 1, s)));
  pfloatx16 t1, t2, t3;
#pragma unroll
  for (int v = 0; v < 16; ++v) t1[v] = t2[v] = t3[v] = 0.f;
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const float4 a = As[(2 * s + half) * 32 + col];
    t1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, x[s].x, t1, 0, 0, 0);
    t2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, x[s].y, t2, 0, 0, 0);
    t3 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, x[s].x + x[s].y, t3, 0, 0, 0);
  }
  // C layout: lane l, register v -> group l%32, amplitude 8(v/4) + 4(l/32) + v%4
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const uint32_t o = xor_bits<2>(b.row, v & 3) ^ xor_bits<2>(b.row + 3, v >> 2);
    *reinterpret_cast<float2 *>(X + (wr ^ o)) = make_float2(t1[v] - t2[v], t3[v] - t1[v] - t2[v]);
  }
}

// A-operand registers of a 4-target block's real 32x32 form.
__device__ __forceinline__ void pass_a4(float (&a)[16], const float *As, int lane) {
#pragma unroll
  for (int s = 0; s < 16; ++s) a[s] = As[(2 * s + (lane >> 5)) * 32 + (lane & 31)];
}
__device__ __forceinline__ void pass_a4(double (&a)[16], const double *As, int lane) {
#pragma unroll
  for (int s = 0; s < 16; ++s) a[s] = As[(4 * (s >> 1) + (lane >> 4)) * 32 + 16 * (s & 1) + (lane & 15)];
}

// One 4-target block on two tiles (complex64): the real 32x32 form, operands
// as in k_mfma4_c64.
__device__ __forceinline__ void pass_block4(char *X, const float (&a)[16], const PassBlock &b,
                                            int lane, uint32_t lb, uint32_t tile2) {
  const int half = lane >> 5;
  float x0[16], x1[16];
  const uint32_t rd = lb | (half ? 4u : 0u);
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const uint32_t o = xor_bits<4>(b.row, s);
    x0[s] = *reinterpret_cast<const float *>(X + (rd ^ o));
    x1[s] = *reinterpret_cast<const float *>(X + (rd ^ o ^ tile2));
  }
  pfloatx16 t0, t1;
#pragma unroll
  for (int v = 0; v < 16; ++v) t0[v] = t1[v] = 0.f;
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    t0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], x0[s], t0, 0, 0, 0);
    t1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], x1[s], t1, 0, 0, 0);
  }
  // C layout: lane l, register 4q + i -> component i%2 of amplitude 4q + 2(l/32) + i/2
  const uint32_t wr = lb ^ (half ? b.row[1] : 0u);
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t o = xor_bits<2>(b.row + 2, q) ^ (i ? b.row[0] : 0u);
      *reinterpret_cast<float2 *>(X + (wr ^ o)) = make_float2(t0[4 * q + 2 * i], t0[4 * q + 2 * i + 1]);
      *reinterpret_cast<float2 *>(X + (wr ^ o ^ tile2)) =
          make_float2(t1[4 * q + 2 * i], t1[4 * q + 2 * i + 1]);
    }
}

// complex128 forms (v_mfma_f64_16x16x4f64), operands as in k_mfma5_c128 and
// k_mfma4_c128.
__device__ __forceinline__ void pass_block5(char *X, const double2 *As, const PassBlock &b,
                                            int lane, uint32_t lb) {
  const int col = lane & 15, q = lane >> 4;
  const uint32_t rd = lb ^ xor_lane<2>(b.row, q);
  double2 x[8];
#pragma unroll
  for (int s = 0; s < 8; ++s)
    x[s] = *reinterpret_cast<const double2 *>(X + (rd ^ xor_bits<3>(b.row + 2, s)));
  pdoublex4 t1[2], t2[2], t3[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) t1[t][v] = t2[t][v] = t3[t][v] = 0.0;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const double xs = x[s].x + x[s].y;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const double2 a = As[(4 * s + q) * 32 + 16 * t + col];
      t1[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x[s].x, t1[t], 0, 0, 0);
      t2[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, x[s].y, t2[t], 0, 0, 0);
      t3[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x + a.y, xs, t3[t], 0, 0, 0);
    }
  }
  // C layout: lane l, register v of block t -> group l%16, amplitude 16t + 4v + l/16
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const uint32_t o = xor_bits<2>(b.row + 2, v) ^ (t ? b.row[4] : 0u);
      *reinterpret_cast<double2 *>(X + (rd ^ o)) =
          make_double2(t1[t][v] - t2[t][v], t3[t][v] - t1[t][v] - t2[t][v]);
    }
}

__device__ __forceinline__ void pass_block4(char *X, const double (&a)[16], const PassBlock &b,
                                            int lane, uint32_t lb, uint32_t tile2) {
  const int q = lane >> 4;
  const uint32_t rd = (lb ^ ((q >> 1) ? b.row[0] : 0u)) | ((q & 1) ? 8u : 0u);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    double x[8];
#pragma unroll
    for (int s = 0; s < 8; ++s)
      x[s] = *reinterpret_cast<const double *>(X + (rd ^ xor_bits<3>(b.row + 1, s) ^ (h ? tile2 : 0u)));
    pdoublex4 acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[t][v] = 0.0;
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[2 * s + t], x[s], acc[t], 0, 0, 0);
    // C layout: lane l, register v of block t -> component (l/16)%2 of
    // amplitude 8t + 2v + (l/16)/2
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const uint32_t o = xor_bits<2>(b.row + 1, v) ^ (t ? b.row[3] : 0u) ^ (h ? tile2 : 0u);
        *reinterpret_cast<double *>(X + (rd ^ o)) = acc[t][v];
      }
  }
}

// A block descriptor in scalar registers (whole dwords: there are no 16-bit
// scalar loads).
__device__ __forceinline__ PassBlock load_block(const PassBlock *p) {
  uint32_t w[sizeof(PassBlock) / 4];
#pragma unroll
  for (int i = 0; i < (int)(sizeof(PassBlock) / 4); ++i)
    w[i] = __builtin_amdgcn_readfirstlane(reinterpret_cast<const uint32_t *>(p)[i]);
  PassBlock b;
  __builtin_memcpy(&b, w, sizeof(b));
  return b;
}

// Launch shape of a chunk size: waves per workgroup and 16-byte accesses per
// thread.
template <typename R, int CB>
struct PassShape {
  static constexpr int NW = 1 << (CB - (sizeof(R) == 4 ? 10 : 9));  // one 5-target tile each
  static constexpr int NT = 64 * NW;
  static constexpr int NL = (1 << CB) * (sizeof(R) == 4 ? 8 : 16) / 16 / NT;
};

template <typename R, int CB>
__global__ void __launch_bounds__((PassShape<R, CB>::NT), (PassShape<R, CB>::NW == 8 ? 4 : 2))
    k_pass(typename CV<R>::T *__restrict__ sv, uint64_t sstride, uint64_t nchunks, PassGeom geom,
           const PassBlock *__restrict__ blocks, int nblocks, const char *__restrict__ image,
           uint64_t gstride) {
  using T = typename CV<R>::T;
  using S = PassShape<R, CB>;
  constexpr bool c64 = sizeof(R) == 4;
  constexpr int NT = S::NT, NW = S::NW, NL = S::NL;
  constexpr int WB = CB - (c64 ? 10 : 9);             // wave index bits
  constexpr int TB = 6 + (NW == 8 ? 3 : NW == 4 ? 2 : NW == 2 ? 1 : 0);  // thread index bits
  constexpr int E0 = c64 ? 1 : 0;                     // chunk bit of thread bit 0 (16 B per access)
  constexpr int EK = E0 + TB;                         // chunk bit of access index bit 0
  constexpr int ITEM = c64 ? 8 : 16;
  constexpr int NP = 1024 / NT;                       // 16-byte units of a block matrix per thread
  __shared__ T Xs[1 << CB];
  __shared__ float4 As[1024];
  char *X = reinterpret_cast<char *>(Xs);
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  sv += blockIdx.y * sstride;
  const nt_f4 *G = reinterpret_cast<const nt_f4 *>(image + blockIdx.y * gstride);
  uint64_t la = 0;
  uint32_t tw = 0;
#pragma unroll
  for (int i = 0; i < TB; ++i)
    if ((t >> i) & 1) {
      la += geom.addr[i + E0];
      tw ^= pass_slot<R>(i + E0) * ITEM;
    }
  // address and slot of access k
  auto ka = [&](int k) {
    uint64_t a = 0;
#pragma unroll
    for (int i = 0; i < CB - EK; ++i) a += ((k >> i) & 1) ? geom.addr[EK + i] : 0;
    return a;
  };
  auto kw = [&](int k) {
    uint32_t w = 0;
#pragma unroll
    for (int i = 0; i < CB - EK; ++i) w ^= ((k >> i) & 1) ? pass_slot<R>(EK + i) * ITEM : 0u;
    return w;
  };
  // this thread's units of a block's matrix image (units past its end repeat
  // the last one)
  auto fetch = [&](nt_f4(&pre)[NP], const PassBlock *pb) {
    const PassBlock b = load_block(pb);
    const nt_f4 *g = G + b.goff;
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (i * NT < b.n16) {
        const int u = t + i * NT;
        pre[i] = g[u < b.n16 ? u : b.n16 - 1];
      }
  };
  auto chunk = [&](uint64_t c) {
    uint64_t base = c;
    for (int j = 0; j < geom.nins; ++j) {
      const uint64_t lo = base & geom.lowmask[j];
      base = ((base ^ lo) << 1) | lo;
    }
    return sv + ((base << geom.shift) + la);
  };
  for (uint64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
    T *p = chunk(c);
    nt_f4 v[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k)
      v[k] = __builtin_nontemporal_load(reinterpret_cast<const nt_f4 *>(p + ka(k)));
    nt_f4 pre[NP];
    fetch(pre, blocks);
    if (c != blockIdx.x) __syncthreads();  // the last chunk has been read out
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      if constexpr (c64) {
        *reinterpret_cast<float2 *>(X + (tw ^ kw(k))) = make_float2(v[k].x, v[k].y);
        *reinterpret_cast<float2 *>(X + (tw ^ kw(k) ^ ITEM)) = make_float2(v[k].z, v[k].w);
      } else {
        *reinterpret_cast<nt_f4 *>(X + (tw ^ kw(k))) = v[k];
      }
    }
    for (int j = 0; j < nblocks; ++j) {
      const PassBlock b = load_block(blocks + j);
#pragma unroll
      for (int i = 0; i < NP; ++i)
        if (i * NT < b.n16) reinterpret_cast<nt_f4 *>(As)[t + i * NT] = pre[i];
      __syncthreads();
      if (j + 1 < nblocks) fetch(pre, blocks + j + 1);  // arrives during this block's products
      uint32_t lb = xor_lane<c64 ? 5 : 4>(b.col, lane);
      lb ^= xor_lane<WB>(b.wave, wave);
      if (b.k == 5) {
        if constexpr (c64) pass_block5(X, As, b, lane, lb);
        else pass_block5(X, reinterpret_cast<const double2 *>(As), b, lane, lb);
      } else {
        R a[16];
        pass_a4(a, reinterpret_cast<const R *>(As), lane);
        pass_block4(X, a, b, lane, lb, b.wave[WB]);
      }
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      nt_f4 o;
      if constexpr (c64) {
        const float2 y0 = *reinterpret_cast<const float2 *>(X + (tw ^ kw(k)));
        const float2 y1 = *reinterpret_cast<const float2 *>(X + (tw ^ kw(k) ^ ITEM));
        o = nt_f4{y0.x, y0.y, y1.x, y1.y};
      } else {
        o = *reinterpret_cast<const nt_f4 *>(X + (tw ^ kw(k)));
      }
      __builtin_nontemporal_store(o, reinterpret_cast<nt_f4 *>(p + ka(k)));
    }
  }
}

template <typename R, int CB>
static void launch_pass_cb(const PassGeom &geom, void *sv, uint64_t nelems, uint32_t nsets,
                           const PassBlock *blocks, int nblocks, const void *image,
                           uint64_t gstride, hipStream_t st) {
  const uint64_t nchunks = nelems >> CB;
  const uint64_t g = std::min<uint64_t>(nchunks, kPassGrid);
  hipLaunchKernelGGL((k_pass<R, CB>), dim3((unsigned)g, nsets), dim3(PassShape<R, CB>::NT), 0, st,
                     (typename CV<R>::T *)sv, nelems, nchunks, geom, blocks, nblocks,
                     (const char *)image, gstride);
}

int launch_pass(const PassPlan &p, const PassGeom &geom, sq_dtype_t dt, void *sv,
                uint64_t nelems, uint32_t nsets, const PassBlock *blocks, int nblocks,
                const void *image, uint64_t gstride, hipStream_t st) {
  if (nelems < (1ull << p.cb) || nblocks < 1 || nsets < 1 || nsets > 65535 || !blocks || !image)
    return fail(SQ_ERR_INVALID, "internal: pass does not fit the state");
#define SQ_PASS(R, CB) \
  launch_pass_cb<R, CB>(geom, sv, nelems, nsets, blocks, nblocks, image, gstride, st)
  if (dt == SQ_COMPLEX64) {
    switch (p.cb) {
      case 10: SQ_PASS(float, 10); break;
      case 11: SQ_PASS(float, 11); break;
      case 12: SQ_PASS(float, 12); break;
      case 13: SQ_PASS(float, 13); break;
      default: return fail(SQ_ERR_INVALID, "internal: pass chunk size");
    }
  } else {
    switch (p.cb) {
      case 9: SQ_PASS(double, 9); break;
      case 10: SQ_PASS(double, 10); break;
      case 11: SQ_PASS(double, 11); break;
      case 12: SQ_PASS(double, 12); break;
      default: return fail(SQ_ERR_INVALID, "internal: pass chunk size");
    }
  }
#undef SQ_PASS
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}

}  // namespace sq
