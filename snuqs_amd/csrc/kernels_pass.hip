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
// Bound: the sweep takes 2.7 ms of HBM time at 2^30 complex64 amplitudes at copy
// rate; a complex64 5-target block 0.7 ms of bf16 MFMA at 2.4 GHz (1.3 ms on
// the FP32 instructions), and the clock falls with the matrix work (2.4 GHz
// with none, 2.0 with two blocks, 1.7 with four).  Measured there, local bits
// 0-3, 6, 10, 12, ..., 28: no block 3.5 ms, 1 block 3.6, 2 blocks 3.9, 3 blocks
// 4.9, 4 blocks 6.1 (FP32 instructions: 3.4, 3.6, 4.7, 5.9, 7.4), where one
// block per launch takes 3.1 ms each.  Layered 30-qubit circuit of depth 10 in
// 48 blocks: 148 -> 71-80 ms by box; 25-qubit mixed circuit of 175 gates unfused: 12.4 ->
// 1.1 ms.  A loop over several chunks per workgroup with the next chunk's loads
// issued ahead of the products (4 waves, 2 tiles each) measured 5-10% slower
// than one chunk per workgroup: the two workgroups of a CU already overlap
// one's loads with the other's products.
#include <algorithm>

#include "kernels.hpp"
#include "pass_plan.hpp"

namespace sq {

// Workgroups of a pass in x (one chunk each), since a dimension holds fewer than
// 2^32 work-items; the rest go to z, or to further launches (circuit batches).
constexpr uint64_t kPassGrid = 1ull << 22;

// 16 bytes of a state, which starts at any of its elements' boundaries (the
// accesses are global_load / store_dwordx4, which ask for no more than dwords).
typedef float state_f4 __attribute__((ext_vector_type(4), aligned(4)));
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

// complex64 products run on the bf16 matrix instructions (16 times the FP32
// rate) with every FP32 operand split in three bf16 parts: the six products of
// parts i + j <= 2 are summed in FP32.  Each part is a nearest 8-bit value, so |x1|
// <= 2^-8 |x0| and |x2| <= 2^-17 |x0|: x0 + x1 + x2 is x (24 bits), or the FP64
// matrix entry to 2^-26, and a sum of six products is within 2^-24 of g x (the
// bound of an FP32 product's rounding), 2^-27 root mean square over random
// operands.  Parts are exact for |x| from 2^-108 (below, x2 is subnormal) to
// 3.396e38 (above, x0 is infinite).
// The matrix parts come from its FP64 entries (pass_image).  Error of a layered
// circuit against 64 bits (2-norm): 14 qubits 6.3e-7 -> 3.6e-7, 23 qubits 7.4e-7
// -> 4.3e-7, 30 qubits 7.9e-7 -> 4.7e-7 against the FP32 instructions with three
// real products per complex one.
typedef __bf16 pbf2 __attribute__((ext_vector_type(2)));
typedef __bf16 pbf8 __attribute__((ext_vector_type(8)));
typedef float pf2 __attribute__((ext_vector_type(2)));

// Parts of eight operands of this lane.
struct Split8 {
  pbf8 p[3];
};
__device__ __forceinline__ void split2(Split8 &s, int i, float a, float b) {
  pf2 x = {a, b};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const pbf2 h = __builtin_convertvector(x, pbf2);
    s.p[k][2 * i] = h[0];
    s.p[k][2 * i + 1] = h[1];
    if (k < 2) {
      const pf2 f = __builtin_convertvector(h, pf2);
      x[0] -= f[0];
      x[1] -= f[1];
    }
  }
}
// One 5-target block on this wave's tile (complex64): T1 = Gr Xr, T2 = Gi Xi,
// T3 = Gi Xr + Gr Xi.  Fragment (m, part, t) of the matrix image (m = 0: Gr,
// 1: Gi) holds lane l's G[l%32][16t + 8(l/32) + j], j = 0..7; the state operand
// of lane l is amplitude 16t + 8(l/32) + j of group l%32.
__device__ __forceinline__ void pass_block5(char *X, const pbf8 *As, const PassBlock &b, int lane,
                                            uint32_t lb) {
  const int half = lane >> 5;
  const uint32_t rd = lb ^ (half ? b.row[3] : 0u), wr = lb ^ (half ? b.row[2] : 0u);
  pfloatx16 t1, t2, t3;
#pragma unroll
  for (int v = 0; v < 16; ++v) t1[v] = t2[v] = t3[v] = 0.f;
  float2 u[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j)
      u[t][j] = *reinterpret_cast<const float2 *>(
          X + (rd ^ (t ? b.row[4] : 0u) ^ xor_bits<3>(b.row, j)));
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    Split8 xr, xi;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      split2(xr, i, u[t][2 * i].x, u[t][2 * i + 1].x);
      split2(xi, i, u[t][2 * i].y, u[t][2 * i + 1].y);
    }
    // part p of the matrix against parts 2 - p, ..., 0 of the state
#pragma unroll
    for (int p = 2; p >= 0; --p) {
      const pbf8 gr = As[(2 * p + t) * 64 + lane], gi = As[(2 * (3 + p) + t) * 64 + lane];
#pragma unroll
      for (int x = 2 - p; x >= 0; --x) {
        t1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gr, xr.p[x], t1, 0, 0, 0);
        t3 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gi, xr.p[x], t3, 0, 0, 0);
        t2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gi, xi.p[x], t2, 0, 0, 0);
        t3 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gr, xi.p[x], t3, 0, 0, 0);
      }
    }
  }
  // C layout: lane l, register v -> group l%32, amplitude 8(v/4) + 4(l/32) + v%4
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const uint32_t o = xor_bits<2>(b.row, v & 3) ^ xor_bits<2>(b.row + 3, v >> 2);
    *reinterpret_cast<float2 *>(X + (wr ^ o)) = make_float2(t1[v] - t2[v], t3[v]);
  }
}

// One 4-target block on two tiles (complex64) in its real 32x32 form (row
// 2r + c, column 2o + c').  Fragment (part, t) holds lane l's entries of row
// l%32, columns 16t + 8(l/32) + j; the state operand is component j%2 of
// amplitude 8t + 4(l/32) + j/2.
__device__ __forceinline__ void pass_block4(char *X, const pbf8 *As, const PassBlock &b, int lane,
                                            uint32_t lb, uint32_t tile2) {
  const int half = lane >> 5;
  const uint32_t rd = lb ^ (half ? b.row[2] : 0u);
  pfloatx16 t0, t1;
#pragma unroll
  for (int v = 0; v < 16; ++v) t0[v] = t1[v] = 0.f;
  float2 u[2][4], v[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t o = rd ^ (t ? b.row[3] : 0u) ^ xor_bits<2>(b.row, i);
      u[t][i] = *reinterpret_cast<const float2 *>(X + o);
      v[t][i] = *reinterpret_cast<const float2 *>(X + (o ^ tile2));
    }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    Split8 x0, x1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      split2(x0, i, u[t][i].x, u[t][i].y);
      split2(x1, i, v[t][i].x, v[t][i].y);
    }
#pragma unroll
    for (int p = 2; p >= 0; --p) {
      const pbf8 g = As[(2 * p + t) * 64 + lane];
#pragma unroll
      for (int x = 2 - p; x >= 0; --x) {
        t0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g, x0.p[x], t0, 0, 0, 0);
        t1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g, x1.p[x], t1, 0, 0, 0);
      }
    }
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

__device__ __forceinline__ void pass_block4(char *X, const double *As, const PassBlock &b, int lane,
                                            uint32_t lb, uint32_t tile2) {
  const int q = lane >> 4;
  double a[16];
#pragma unroll
  for (int s = 0; s < 16; ++s) a[s] = As[(4 * (s >> 1) + q) * 32 + 16 * (s & 1) + (lane & 15)];
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
struct PassLds {
  typename CV<R>::T x[1 << CB];
  float4 a[sizeof(R) == 4 ? 768 : 1024];
};

// The pass on chunk c of a state: by every thread of the workgroup.  initial:
// the state is |0...0> and is not read.  STREAM: non-temporal accesses.
template <typename R, int CB, bool STREAM>
__device__ __forceinline__ void pass_chunk(typename CV<R>::T *__restrict__ sv, uint64_t c,
                                           const PassGeom &geom,
                                           const PassBlock *__restrict__ blocks, int nblocks,
                                           const nt_f4 *__restrict__ G, bool initial,
                                           PassLds<R, CB> &lds) {
  using S = PassShape<R, CB>;
  constexpr bool c64 = sizeof(R) == 4;
  constexpr int NT = S::NT, NW = S::NW, NL = S::NL;
  constexpr int WB = CB - (c64 ? 10 : 9);             // wave index bits
  constexpr int TB = 6 + WB;                          // thread index bits
  constexpr int E0 = c64 ? 1 : 0;                     // chunk bit of thread bit 0 (16 B per access)
  constexpr int EK = E0 + TB;                         // chunk bit of access index bit 0
  constexpr int ITEM = c64 ? 8 : 16;
  constexpr int NP = (c64 ? 768 + NT - 1 : 1024) / NT;  // 16-byte units of a block matrix per thread
  static_assert(NW == 1 << WB, "one wave a tile");
  char *X = reinterpret_cast<char *>(lds.x);
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
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
  uint64_t base = c;
  for (int j = 0; j < geom.nins; ++j) {
    const uint64_t lo = base & geom.lowmask[j];
    base = ((base ^ lo) << 1) | lo;
  }
  typename CV<R>::T *p = sv + ((base << geom.shift) + la);
  nt_f4 v[NL];
  if (initial) {
#pragma unroll
    for (int k = 0; k < NL; ++k) v[k] = nt_f4{0.f, 0.f, 0.f, 0.f};
    if (c != 0) {  // stays zero
#pragma unroll
      for (int k = 0; k < NL; ++k)
        __builtin_nontemporal_store((state_f4)v[k], reinterpret_cast<state_f4 *>(p + ka(k)));
      return;
    }
    if (t == 0) {
      if constexpr (c64) {
        v[0].x = 1.f;
      } else {
        const double2 one = make_double2(1.0, 0.0);
        __builtin_memcpy(&v[0], &one, 16);
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const state_f4 *q = reinterpret_cast<const state_f4 *>(p + ka(k));
      if constexpr (STREAM) v[k] = __builtin_nontemporal_load(q);
      else v[k] = *q;
    }
  }
  nt_f4 pre[NP];
  fetch(pre, blocks);
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
      if (t + i * NT < b.n16) reinterpret_cast<nt_f4 *>(lds.a)[t + i * NT] = pre[i];
    __syncthreads();
    if (j + 1 < nblocks) fetch(pre, blocks + j + 1);  // arrives during this block's products
    uint32_t lb = xor_lane<c64 ? 5 : 4>(b.col, lane);
    lb ^= xor_lane<WB>(b.wave, wave);
    if (b.k == 5) {
      if constexpr (c64) pass_block5(X, reinterpret_cast<const pbf8 *>(lds.a), b, lane, lb);
      else pass_block5(X, reinterpret_cast<const double2 *>(lds.a), b, lane, lb);
    } else {
      if constexpr (c64)
        pass_block4(X, reinterpret_cast<const pbf8 *>(lds.a), b, lane, lb, b.wave[WB]);
      else
        pass_block4(X, reinterpret_cast<const double *>(lds.a), b, lane, lb, b.wave[WB]);
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
    state_f4 *q = reinterpret_cast<state_f4 *>(p + ka(k));
    if constexpr (STREAM) __builtin_nontemporal_store((state_f4)o, q);
    else *q = o;
  }
}

#define SQ_PASS_BOUNDS \
  __launch_bounds__((PassShape<R, CB>::NT), \
                    (PassShape<R, CB>::NW == 8 ? 4 : PassShape<R, CB>::NW == 4 ? 3 : 2))

template <typename R, int CB, bool STREAM>
__global__ void SQ_PASS_BOUNDS
    k_pass(typename CV<R>::T *__restrict__ sv, uint64_t sstride, uint64_t nchunks, PassGeom geom,
           const PassBlock *__restrict__ blocks, int nblocks, const char *__restrict__ image,
           uint64_t gstride) {
  __shared__ PassLds<R, CB> lds;
  const nt_f4 *G = reinterpret_cast<const nt_f4 *>(image + blockIdx.y * gstride);
  const uint64_t c = (uint64_t)blockIdx.z * gridDim.x + blockIdx.x;
  if (c < nchunks)
    pass_chunk<R, CB, STREAM>(sv + blockIdx.y * sstride, c, geom, blocks, nblocks, G, false, lds);
}

// Circuit batches: workgroup w of a step takes chunk w - first of its entry
// (this launch's are w0, w0 + 1, ...).
template <typename R, int CB, bool STREAM>
__global__ void SQ_PASS_BOUNDS
    k_pass_entries(typename CV<R>::T *__restrict__ states, const PassEntry *__restrict__ entries,
                   const uint32_t *__restrict__ entry, uint64_t w0,
                   const PassBlock *__restrict__ blocks, const char *__restrict__ images) {
  __shared__ PassLds<R, CB> lds;
  const uint64_t w = w0 + blockIdx.x;
  const PassEntry &e = entries[__builtin_amdgcn_readfirstlane(entry[w])];
  pass_chunk<R, CB, STREAM>(states + e.psi, w - e.first, e.geom, blocks + e.blocks, e.nblocks,
                        reinterpret_cast<const nt_f4 *>(images + e.image), e.initial != 0, lds);
}

// Ordinary instead of non-temporal accesses: states of up to 2 MiB, half of what
// each XCD's L2 holds, and those above what the eight L2s hold together (32 MiB)
// that fit the Infinity Cache (256 MiB).  (In between, a chunk's lines presumably lie
// in the L2 of another XCD, which had them in the last pass.)  Non-temporal over
// ordinary time,
// layered circuits as programs, complex64 / complex128: 128 KiB 1.03-1.04 / 1.04-1.05,
// 1 MiB 1.03-1.04 / 1.02-1.04, 2 MiB 1.03 / 1.03, 4 MiB 1.00-1.01 / 1.00-1.01, 8 MiB
// 0.98-1.00 / 0.96-0.97, 16 MiB 0.94 / 0.86-0.88, 32 MiB 1.01-1.10 / 0.98-0.99, 64 MiB
// 1.02 / 0.98-1.00, 128 MiB 1.06-1.08 / 1.03-1.04, 256 MiB 1.07-1.08 / 1.05-1.07, 512
// MiB 0.99 / 0.98-0.99.  Parameter batches by all their states: up to 2 MiB 1.00, 4-16
// MiB 0.85-0.96, 64-256 MiB 1.01-1.07 / 1.02, 512 MiB 0.98 / 0.99.  Circuit batches: up
// to 2 MiB 1.00-1.02, 8-32 MiB 0.79-0.99, 64-128 MiB 1.02-1.05 / 0.98-0.99, 256 MiB
// 0.99 / 0.99: complex128 ones stay non-temporal above 2 MiB.
// The choice is a template argument: the compiler merges accesses that differ
// in this hint alone.
static bool pass_cached(uint64_t bytes) {
  return bytes <= 2ull << 20 || (bytes > 32ull << 20 && bytes <= 256ull << 20);
}

template <typename R, int CB>
static void launch_pass_cb(const PassGeom &geom, void *sv, uint64_t nelems, uint32_t nsets,
                           const PassBlock *blocks, int nblocks, const void *image,
                           uint64_t gstride, hipStream_t st) {
  const uint64_t nchunks = nelems >> CB;
  const uint64_t g = std::min<uint64_t>(nchunks, kPassGrid);
  const auto k = pass_cached(nelems * nsets * sizeof(typename CV<R>::T)) ? k_pass<R, CB, false>
                                                                         : k_pass<R, CB, true>;
  hipLaunchKernelGGL(k, dim3((unsigned)g, nsets, (unsigned)((nchunks + g - 1) / g)), dim3(PassShape<R, CB>::NT), 0, st,
                     (typename CV<R>::T *)sv, nelems, nchunks, geom, blocks, nblocks,
                     (const char *)image, gstride);
}

// SQ_PASS(R, CB) for the dtype and chunk size.
#define SQ_PASS_SWITCH(cb)                                                      \
  switch ((dt == SQ_COMPLEX64 ? 0 : 100) + (cb)) {                              \
    case 10: SQ_PASS(float, 10); break;                                         \
    case 11: SQ_PASS(float, 11); break;                                         \
    case 12: SQ_PASS(float, 12); break;                                         \
    case 13: SQ_PASS(float, 13); break;                                         \
    case 109: SQ_PASS(double, 9); break;                                        \
    case 110: SQ_PASS(double, 10); break;                                       \
    case 111: SQ_PASS(double, 11); break;                                       \
    case 112: SQ_PASS(double, 12); break;                                       \
    default: return fail(SQ_ERR_INVALID, "internal: pass chunk size");          \
  }

uint64_t pass_entry_launches(uint64_t nwg) { return (nwg + kPassGrid - 1) / kPassGrid; }

int launch_pass_entries(int cb, sq_dtype_t dt, void *states, const PassEntry *entries,
                        const uint32_t *entry, const PassBlock *blocks, const void *images,
                        uint64_t nwg, hipStream_t st) {
  const uint64_t bytes = (nwg << cb) * itemsize(dt);
  const bool cached = pass_cached(bytes) && (dt == SQ_COMPLEX64 || bytes <= 2ull << 20);
#define SQ_PASS(R, CB)                                                                          \
  hipLaunchKernelGGL((cached ? k_pass_entries<R, CB, false> : k_pass_entries<R, CB, true>),     \
                     dim3((unsigned)std::min(nwg - w0, kPassGrid)), dim3(PassShape<R, CB>::NT), \
                     0, st, (typename CV<R>::T *)states, entries, entry, w0, blocks,            \
                     (const char *)images)
  for (uint64_t w0 = 0; w0 < nwg; w0 += kPassGrid) {
    SQ_PASS_SWITCH(cb)
    SQ_HIP(hipGetLastError());
  }
#undef SQ_PASS
  return SQ_OK;
}

int launch_pass(const PassPlan &p, const PassGeom &geom, sq_dtype_t dt, void *sv,
                uint64_t nelems, uint32_t nsets, const PassBlock *blocks, int nblocks,
                const void *image, uint64_t gstride, hipStream_t st) {
  if (nelems < (1ull << p.cb) || nblocks < 1 || nsets < 1 || nsets > 65535 || !blocks || !image)
    return fail(SQ_ERR_INVALID, "internal: pass does not fit the state");
#define SQ_PASS(R, CB) \
  launch_pass_cb<R, CB>(geom, sv, nelems, nsets, blocks, nblocks, image, gstride, st)
  SQ_PASS_SWITCH(p.cb)
#undef SQ_PASS
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}

}  // namespace sq
