// kernels_cbatch.hip -- circuits of uneven qubit counts and different gate
// lists run as one launch sequence.
//
// No reference counterpart (the reference runs one circuit per simulation and
// has no batching; transpile.py:233-234 is where it would go).  Circuit j has
// n_j qubits and its own list of gates (dense matrices on 1-5 targets, e.g.
// the blocks of a fused circuit); its state lives at its own offset in one
// device buffer.
//
// Circuits large enough for a pass (kernels_pass.hip) are planned into passes
// of several gates; launch s applies pass s of every such circuit, one
// workgroup a chunk, a table giving each workgroup its circuit.  A circuit's
// first pass starts from |0...0> without reading it.  Smaller circuits take
// gate s of each in one launch of k_cbatch_dense.  So many small circuits,
// each of which alone would leave most of the GPU idle, fill it together, and
// a batch takes as many launches as its longest circuit has steps (captured in
// one hipGraph).  48 circuits of 12-22 qubits, depth 10, complex64: 4.2 ms a
// run with one gate a step, 1.7 ms with passes.
//
// k_cbatch_dense: a group is the 2^k amplitudes a k-target gate mixes; one lane
// per group per grid pass, consecutive lanes on consecutive groups (coalesced
// runs along the lowest free bits); the matrix is staged in LDS, so every lane
// of a wave reads the same entry (a broadcast).  Arithmetic in the state's
// precision.
#include <algorithm>
#include <cstring>
#include <memory>
#include <new>
#include <vector>

#include "kernels.hpp"
#include "kernels_cbatch.hpp"
#include "pass_plan.hpp"

namespace sq {

// One gate of one circuit within a launch.
struct CBGate {
  uint64_t psi;          // amplitude offset of the circuit's state
  uint64_t nfree;        // groups: 2^(n - k)
  uint64_t first_block;  // first workgroup of the gate in its launch
  uint64_t nblocks;      // its workgroups (grid stride over its groups)
  uint64_t mat;          // element offset of its matrix (plan order, row-major)
  IdxMap im;             // group index -> amplitude index (target bits 0)
  int k, pad0, pad1, pad2;
  int tb[kMaxK];         // amplitude bit of target b (local index bit b)
  int pad3[8 - kMaxK];
};

// The entry whose workgroup range holds workgroup b (first_block ascending).
// With at most kBlock entries their first blocks are staged in LDS by one
// load per thread and searched there.  Every thread must call it.
__device__ __forceinline__ int cb_find(const CBGate *tab, int count, uint64_t b) {
  __shared__ uint64_t sfb[kBlock];
  int lo = 0, hi = count - 1;
  if (count > kBlock) {
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (tab[mid].first_block <= b) lo = mid; else hi = mid - 1;
    }
  } else {
    if ((int)threadIdx.x < count) sfb[threadIdx.x] = tab[threadIdx.x].first_block;
    __syncthreads();
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (sfb[mid] <= b) lo = mid; else hi = mid - 1;
    }
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// y = M x on every group of the gate assigned to this workgroup.  M is
// staged in LDS as (re, im) pairs, row-major (a complex64 row is read two
// entries per 16-byte access), after the workgroup's first groups are
// requested: the two latencies overlap.  A group's amplitude offsets come
// from the target bits (uniform), so no table sits between the entry and
// the loads.  Every thread of the workgroup must call it (it synchronises).
template <typename R, int K>
__device__ __forceinline__ void cb_body(typename CV<R>::T *__restrict__ sv, const CBGate &g,
                                        uint64_t wg, const typename CV<R>::T *__restrict__ mat,
                                        typename CV<R>::T *M) {
  using T = typename CV<R>::T;
  constexpr int D = 1 << K;
  int tb[K];
#pragma unroll
  for (int b = 0; b < K; ++b) tb[b] = g.tb[b];
  auto offc = [&](int c) {
    uint64_t o = 0;
#pragma unroll
    for (int b = 0; b < K; ++b)
      if ((c >> b) & 1) o += 1ull << tb[b];
    return o;
  };
  const uint64_t stride = g.nblocks * kBlock;
  uint64_t f = wg * kBlock + threadIdx.x;
  T x[D];
  uint64_t base = 0;
  if (f < g.nfree) {
    base = deposit(f, g.im);
#pragma unroll
    for (int c = 0; c < D; ++c) x[c] = ld_nt(sv + base + offc(c));
  }
  for (int e = threadIdx.x; e < D * D; e += kBlock) M[e] = mat[e];
  __syncthreads();
  while (f < g.nfree) {
    // 1-2 targets: rows unrolled; 3-5: one row at a time (the D inputs stay
    // in registers, the row's entries are LDS broadcasts; unrolled rows would
    // hold the whole matrix in registers)
#pragma unroll K <= 2 ? D : 1
    for (int r = 0; r < D; ++r) {
      R yr = 0, yi = 0;
      if constexpr (sizeof(R) == 4) {
        const float4 *m4 = reinterpret_cast<const float4 *>(M + r * D);
#pragma unroll
        for (int c = 0; c < D; c += 2) {
          const float4 m = m4[c / 2];
          yr += m.x * x[c].x - m.y * x[c].y;
          yi += m.x * x[c].y + m.y * x[c].x;
          yr += m.z * x[c + 1].x - m.w * x[c + 1].y;
          yi += m.z * x[c + 1].y + m.w * x[c + 1].x;
        }
      } else {
#pragma unroll
        for (int c = 0; c < D; ++c) {
          const T m = M[r * D + c];
          yr += m.x * x[c].x - m.y * x[c].y;
          yi += m.x * x[c].y + m.y * x[c].x;
        }
      }
      T o;
      o.x = yr;
      o.y = yi;
      st_nt(sv + base + offc(r), o);
    }
    f += stride;
    if (f < g.nfree) {
      base = deposit(f, g.im);
#pragma unroll
      for (int c = 0; c < D; ++c) x[c] = ld_nt(sv + base + offc(c));
    }
  }
}

template <typename R>
__global__ void __launch_bounds__(kBlock)
    k_cbatch_dense(typename CV<R>::T *__restrict__ st, const typename CV<R>::T *__restrict__ mats,
                   const CBGate *__restrict__ tab, int count) {
  using T = typename CV<R>::T;
  constexpr int DM = 1 << kMaxK;
  __shared__ __align__(16) T M[DM * DM];
  const int e = cb_find(tab, count, blockIdx.x);
  const CBGate &g = tab[e];
  T *sv = st + g.psi;
  const T *mat = mats + g.mat;
  const uint64_t wg = blockIdx.x - g.first_block;
  switch (g.k) {
    case 1: cb_body<R, 1>(sv, g, wg, mat, M); break;
    case 2: cb_body<R, 2>(sv, g, wg, mat, M); break;
    case 3: cb_body<R, 3>(sv, g, wg, mat, M); break;
    case 4: cb_body<R, 4>(sv, g, wg, mat, M); break;
    default: cb_body<R, 5>(sv, g, wg, mat, M); break;
  }
}

// Every state <- |0...0>: zero the buffer, then amplitude 0 of each state.
template <typename R>
__global__ void __launch_bounds__(kBlock) k_cbatch_zero(typename CV<R>::T *__restrict__ st,
                                                        uint64_t nelems) {
  using T = typename CV<R>::T;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < nelems;
       i += (uint64_t)gridDim.x * kBlock)
    st_nt(st + i, T{0, 0});
}
template <typename R>
__global__ void __launch_bounds__(kBlock) k_cbatch_basis(typename CV<R>::T *__restrict__ st,
                                                         const uint64_t *__restrict__ psi,
                                                         uint32_t ncirc) {
  using T = typename CV<R>::T;
  const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
  if (j < ncirc) st[psi[j]] = T{1, 0};
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
constexpr uint64_t kCBMaxBlocksPerGate = 1ull << 14;  // grid stride beyond

struct CBatch {
  sq_dtype_t dt;
  uint32_t ncirc = 0;
  std::vector<uint32_t> nq;
  std::vector<uint64_t> host_psi;
  uint64_t nelems = 0;
  void *states = nullptr;
  void *mats = nullptr;       // matrices of k_cbatch_dense
  CBGate *tables = nullptr;
  void *pass = nullptr;       // entries, workgroup map, descriptors and matrices of the passes
  size_t pass_map = 0, pass_desc = 0, pass_img = 0;  // byte offsets in `pass`
  uint64_t *psi = nullptr;
  struct Launch {
    int cb;          // 0: k_cbatch_dense, otherwise a pass launch's chunk bits
    size_t tab_off;  // first entry of `tables`, or first workgroup of the map
    int count;       // entries (k_cbatch_dense)
    uint64_t blocks;
  };
  std::vector<Launch> launches;
  bool zero_first = false;  // some circuit starts from a state in memory
  hipGraphExec_t exec = nullptr;
  hipGraph_t graph = nullptr;
  double state_bytes = 0, traffic_bytes = 0;
};

static void free_cbatch(CBatch *b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  for (void *p : {b->states, b->mats, (void *)b->tables, b->pass, (void *)b->psi})
    if (p) (void)hipFree(p);
  b->states = b->mats = b->pass = nullptr;
  b->tables = nullptr;
  b->psi = nullptr;
}

// Gates of a batch's circuits as dense matrices on exactly their targets.
struct CBInput {
  const double *matrices;
  std::vector<std::vector<GatePlan>> plans;        // [circuit][gate]
  std::vector<std::vector<int>> nt;
  std::vector<std::vector<size_t>> toff, moff;     // in `targets`, in `matrices`
  std::vector<uint32_t> targets;
};

static int cb_malloc(void **ptr, size_t bytes) {
  if (hipMalloc(ptr, std::max<size_t>(bytes, 16)) != hipSuccess) {
    (void)hipGetLastError();
    *ptr = nullptr;
    return fail(SQ_ERR_OOM, "circuit batch: device allocation of " + std::to_string(bytes) +
                                " failed");
  }
  return SQ_OK;
}

// Steps, launches and device data of a batch: circuits large enough run in
// passes if `with_passes`, every circuit gate by gate otherwise.  SQ_ERR_OOM: no
// room on the device or the host; `B` then holds no device data.
static int cbatch_build(CBatch *B, const CBInput &in, bool with_passes) try {
  const sq_dtype_t dt = B->dt;
  const bool c64 = dt == SQ_COMPLEX64;
  const size_t item = itemsize(dt);
  const uint32_t ncirc = B->ncirc;
  const std::vector<uint32_t> &nq = B->nq;
  const auto &plans = in.plans;
  B->launches.clear();
  B->zero_first = false;
  B->traffic_bytes = 0.0;
  // Steps of the circuits that run in passes.  Chunks are chosen by the batch's
  // amplitudes: together the circuits fill the chip as one state of that size
  // would.
  const int nbits = log2u(B->nelems);
  std::vector<std::vector<PassPlan>> passes(ncirc);
  size_t steps = 0;
  for (uint32_t j = 0; j < ncirc; ++j) {
    const int cb = std::min<int>(pass_chunk_bits(dt, nbits), (int)nq[j]);
    const size_t ng = plans[j].size();
    if (!with_passes || cb < pass_min_bits(dt) || ng == 0) {
      B->zero_first = true;
      steps = std::max(steps, ng);
      continue;
    }
    std::vector<uint64_t> masks(ng, 0);
    for (size_t g = 0; g < ng; ++g)
      for (int b = 0; b < plans[j][g].kk; ++b) masks[g] |= 1ull << plans[j][g].tbit[b];
    std::vector<Step> st;
    plan_passes((int)nq[j], cb, dt, masks, false, &st, &passes[j]);
    steps = std::max(steps, passes[j].size());
  }
  // matrices in the state's precision, tables per launch
  std::vector<double> hm;  // interleaved re/im, converted below
  std::vector<CBGate> tabs;
  std::vector<PassEntry> entries;
  std::vector<uint32_t> wgs;
  std::vector<PassBlock> descs;
  std::vector<char> images;
  for (size_t s = 0; s < steps; ++s) {
    CBatch::Launch L{0, tabs.size(), 0, 0};
    for (uint32_t j = 0; j < ncirc; ++j) {
      if (!passes[j].empty() || s >= plans[j].size()) continue;
      const GatePlan &p = plans[j][s];
      CBGate e{};
      e.psi = B->host_psi[j];
      e.k = p.kk;
      e.nfree = 1ull << (nq[j] - p.kk);
      uint64_t tmask = 0;
      for (int b = 0; b < p.kk; ++b) {
        tmask |= 1ull << p.tbit[b];
        e.tb[b] = p.tbit[b];
      }
      e.im = make_idxmap(tmask, 0);
      e.mat = hm.size() / 2;
      for (const cd &z : p.m) {
        hm.push_back(z.real());
        hm.push_back(z.imag());
      }
      e.first_block = L.blocks;
      e.nblocks = std::min<uint64_t>((e.nfree + kBlock - 1) / kBlock, kCBMaxBlocksPerGate);
      L.blocks += e.nblocks;
      L.count++;
      B->traffic_bytes += 2.0 * std::ldexp(1.0, (int)nq[j]) * (double)item;
      tabs.push_back(e);
    }
    if (L.blocks > (uint64_t)INT32_MAX)
      return fail(SQ_ERR_INVALID, "circuit batch: too many circuits for one launch per step");
    if (L.count) B->launches.push_back(L);
    for (int cb = pass_min_bits(dt); cb <= kPassMaxBits; ++cb) {
      CBatch::Launch P{cb, wgs.size(), 0, 0};
      for (uint32_t j = 0; j < ncirc; ++j) {
        if (s >= passes[j].size() || passes[j][s].cb != cb) continue;
        const PassPlan &p = passes[j][s];
        PassEntry e{};
        size_t bytes;
        const std::vector<PassBlock> pb = pass_blocks(p, dt, &bytes);
        e.psi = B->host_psi[j];
        e.first = P.blocks;
        e.blocks = descs.size();
        e.image = images.size();
        e.nblocks = (int)pb.size();
        e.initial = s == 0;
        e.geom = pass_geom(p);
        images.resize(images.size() + bytes);
        pass_image(p, pb, dt,
                   PassGates{in.matrices, &in.moff[j], &in.toff[j], &in.targets, &in.nt[j], (int)nq[j]},
                   images.data() + e.image);
        descs.insert(descs.end(), pb.begin(), pb.end());
        const uint64_t chunks = 1ull << (nq[j] - cb);
        wgs.insert(wgs.end(), chunks, (uint32_t)entries.size());
        P.blocks += chunks;
        // the first pass writes the state, the others read it too
        B->traffic_bytes += (e.initial ? 1.0 : 2.0) * std::ldexp(1.0, (int)nq[j]) * (double)item;
        entries.push_back(e);
      }
      if (P.blocks) B->launches.push_back(P);
    }
  }
  if (B->zero_first) B->traffic_bytes += (double)B->nelems * (double)item;
  std::vector<char> pimg;
  auto put = [&](const void *src, size_t bytes) {
    const size_t off = (pimg.size() + 255) / 256 * 256;
    pimg.resize(off + bytes);
    if (bytes) std::memcpy(pimg.data() + off, src, bytes);
    return off;
  };
  put(entries.data(), entries.size() * sizeof(PassEntry));
  B->pass_map = put(wgs.data(), wgs.size() * sizeof(uint32_t));
  B->pass_desc = put(descs.data(), descs.size() * sizeof(PassBlock));
  B->pass_img = put(images.data(), images.size());
  const size_t nm = hm.size() / 2;
  int rc = cb_malloc(&B->states, B->nelems * item);
  if (!rc) rc = cb_malloc(&B->mats, nm * item);
  if (!rc) rc = cb_malloc((void **)&B->tables, tabs.size() * sizeof(CBGate));
  if (!rc) rc = cb_malloc(&B->pass, pimg.size());
  if (!rc) rc = cb_malloc((void **)&B->psi, ncirc * sizeof(uint64_t));
  if (rc) {
    free_cbatch(B);
    return rc;
  }
  bool ok = true;
  if (c64) {
    std::vector<float> hf(hm.begin(), hm.end());
    ok = hipMemcpy(B->mats, hf.data(), hf.size() * sizeof(float), hipMemcpyHostToDevice) ==
         hipSuccess;
  } else {
    ok = hipMemcpy(B->mats, hm.data(), hm.size() * sizeof(double), hipMemcpyHostToDevice) ==
         hipSuccess;
  }
  ok = ok && (tabs.empty() || hipMemcpy(B->tables, tabs.data(), tabs.size() * sizeof(CBGate),
                                        hipMemcpyHostToDevice) == hipSuccess);
  ok = ok && (pimg.empty() || hipMemcpy(B->pass, pimg.data(), pimg.size(),
                                        hipMemcpyHostToDevice) == hipSuccess);
  ok = ok && hipMemcpy(B->psi, B->host_psi.data(), ncirc * sizeof(uint64_t),
                       hipMemcpyHostToDevice) == hipSuccess;
  if (!ok) {
    free_cbatch(B);
    return fail(SQ_ERR_HIP, "circuit batch: upload failed");
  }
  return SQ_OK;
} catch (const std::bad_alloc &) {
  free_cbatch(B);
  return fail(SQ_ERR_OOM, "circuit batch: no host memory for its tables");
}

int cbatch_create(void **handle, sq_dtype_t dt, uint32_t ncirc, const uint32_t *nq,
                  const uint32_t *ng, const uint32_t *nt, const uint32_t *targets,
                  const double *matrices) {
  if (ncirc == 0) return fail(SQ_ERR_INVALID, "circuit batch: no circuits");
  auto B = std::make_unique<CBatch>();
  B->dt = dt;
  B->ncirc = ncirc;
  const size_t item = itemsize(dt);
  CBInput in;
  in.matrices = matrices;
  in.plans.resize(ncirc);
  in.nt.resize(ncirc);
  in.toff.resize(ncirc);
  in.moff.resize(ncirc);
  size_t gi = 0, ti = 0, mi = 0;
  uint64_t amp = 0;
  for (uint32_t j = 0; j < ncirc; ++j) {
    if (nq[j] < 1 || nq[j] > 30)
      return fail(SQ_ERR_INVALID, "circuit batch: qubit counts must be in [1, 30]");
    in.plans[j].resize(ng[j]);
    for (uint32_t g = 0; g < ng[j]; ++g, ++gi) {
      const int k = (int)nt[gi];
      if (k < 1 || k > kMaxK || k > (int)nq[j])
        return fail(SQ_ERR_INVALID, "circuit batch: circuit " + std::to_string(j) + ", gate " +
                                        std::to_string(g) + ": 1 to 5 targets, at most the qubit count");
      SQ_TRY(make_plan(matrices + mi, targets + ti, k, (int)nq[j], (int)nq[j], &in.plans[j][g],
                       kPlanDense | kPlanExact));
      if (in.plans[j][g].kind != Kind::DENSE || in.plans[j][g].kk != k)
        return fail(SQ_ERR_INVALID, "circuit batch: internal: gate not planned dense");
      in.nt[j].push_back(k);
      in.toff[j].push_back(ti);
      in.moff[j].push_back(mi);
      ti += (size_t)k;
      mi += 2ull << (2 * k);
    }
    B->nq.push_back(nq[j]);
    B->host_psi.push_back(amp);
    amp += 1ull << nq[j];
    B->state_bytes += std::ldexp(1.0, (int)nq[j]) * (double)item;
  }
  in.targets.assign(targets, targets + ti);
  B->nelems = amp;
  // (the passes' matrices, 6 KiB or more a block, can be what does not fit)
  int rc = cbatch_build(B.get(), in, true);
  if (rc == SQ_ERR_OOM) rc = cbatch_build(B.get(), in, false);
  if (rc != SQ_OK) return rc;
  *handle = B.release();
  return SQ_OK;
}

template <typename R>
static int cb_enqueue_t(CBatch *B, hipStream_t st) {
  using T = typename CV<R>::T;
  T *s = (T *)B->states;
  if (B->zero_first) {  // (a circuit's passes start from |0...0> by themselves)
    const uint64_t zb = std::min<uint64_t>((B->nelems + kBlock - 1) / kBlock, 1ull << 16);
    hipLaunchKernelGGL(k_cbatch_zero<R>, dim3((unsigned)zb), dim3(kBlock), 0, st, s, B->nelems);
    hipLaunchKernelGGL(k_cbatch_basis<R>, dim3((B->ncirc + kBlock - 1) / kBlock), dim3(kBlock), 0,
                       st, s, B->psi, B->ncirc);
  }
  const char *d = (const char *)B->pass;
  for (auto &L : B->launches) {
    if (L.cb)
      SQ_TRY(launch_pass_entries(L.cb, B->dt, B->states, (const PassEntry *)d,
                                 (const uint32_t *)(d + B->pass_map) + L.tab_off,
                                 (const PassBlock *)(d + B->pass_desc), d + B->pass_img, L.blocks,
                                 st));
    else
      hipLaunchKernelGGL(k_cbatch_dense<R>, dim3((unsigned)L.blocks), dim3(kBlock), 0, st, s,
                         (const T *)B->mats, B->tables + L.tab_off, L.count);
  }
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}

static int cb_enqueue(CBatch *B, hipStream_t st) {
  return B->dt == SQ_COMPLEX64 ? cb_enqueue_t<float>(B, st) : cb_enqueue_t<double>(B, st);
}

int cbatch_run(void *handle, int use_graph, hipStream_t st) {
  CBatch *B = (CBatch *)handle;
  if (!use_graph) return cb_enqueue(B, st);
  if (!B->exec) {
    hipStream_t cs;
    SQ_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    int rc = SQ_OK;
    if (hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess)
      rc = fail(SQ_ERR_HIP, "circuit batch: hipStreamBeginCapture failed");
    if (!rc) rc = cb_enqueue(B, cs);
    hipGraph_t g = nullptr;
    if (hipStreamEndCapture(cs, &g) != hipSuccess && !rc)
      rc = fail(SQ_ERR_HIP, "circuit batch: hipStreamEndCapture failed");
    (void)hipStreamDestroy(cs);
    if (rc) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    B->graph = g;
    SQ_HIP(hipGraphInstantiate(&B->exec, g, nullptr, nullptr, 0));
  }
  SQ_HIP(hipGraphLaunch(B->exec, st));
  return SQ_OK;
}

int cbatch_copy_state(void *handle, uint32_t circuit, void *dst, uint64_t nelems,
                      hipStream_t st) {
  CBatch *B = (CBatch *)handle;
  if (circuit >= B->ncirc) return fail(SQ_ERR_INVALID, "circuit batch: no such circuit");
  if (nelems != (1ull << B->nq[circuit]))
    return fail(SQ_ERR_INVALID, "circuit batch: destination has " + std::to_string(nelems) +
                                    " elements, circuit " + std::to_string(circuit) + " has 2^" +
                                    std::to_string(B->nq[circuit]));
  const size_t item = itemsize(B->dt);
  SQ_HIP(hipMemcpyAsync(dst, (const char *)B->states + B->host_psi[circuit] * item,
                        nelems * item, hipMemcpyDeviceToDevice, st));
  return SQ_OK;
}

int cbatch_stats(void *handle, uint64_t *launches, double *state_bytes, double *traffic_bytes) {
  CBatch *B = (CBatch *)handle;
  if (launches) {
    *launches = B->zero_first ? 2 : 0;  // the two initial-state kernels
    for (const auto &L : B->launches) *launches += L.cb ? pass_entry_launches(L.blocks) : 1;
  }
  if (state_bytes) *state_bytes = B->state_bytes;
  if (traffic_bytes) *traffic_bytes = B->traffic_bytes;
  return SQ_OK;
}

int cbatch_destroy(void *handle) {
  CBatch *B = (CBatch *)handle;
  if (!B) return SQ_OK;
  free_cbatch(B);
  delete B;
  return SQ_OK;
}

}  // namespace sq
