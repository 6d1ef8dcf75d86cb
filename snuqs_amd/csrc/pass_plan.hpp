// pass_plan.hpp -- grouping of a gate list into multi-gate passes.
//
// A pass applies several gates of a program in one sweep over the state: a
// workgroup holds a chunk of 2^cb amplitudes (the pass's local bits vary, the
// others are fixed) in LDS, applies every gate of the pass there and writes
// the chunk back, so the state crosses HBM once per pass instead of once per
// gate.  No reference counterpart (the reference sweeps the state once per
// gate, gate_operations_impl_cuda.cu:13-175).
#pragma once

#include <cstdint>
#include <vector>

#include "sq_common.hpp"

namespace sq {

constexpr int kPassMaxBits = 13;  // largest chunk: 2^13 complex64 amplitudes = 64 KiB of LDS

// One matrix of a pass: the product of `gates` (program order) on the state
// bits bits[0..k-1] (ascending, k = 4 or 5).
struct PassBlockPlan {
  int k = 0;
  int bits[kMaxK] = {0};
  std::vector<int> gates;
};

struct PassPlan {
  uint64_t local = 0;  // state bits that vary inside a chunk
  int cb = 0;          // their number
  std::vector<int> gates;  // in an order that gives the same product
  std::vector<PassBlockPlan> blocks;
};

// A program as a sequence of steps: one gate on its own kernel, or one pass.
struct Step {
  int gate = -1;
  int pass = -1;
};

// Smallest chunk (one 5-target tile) and the chunk for launches over 2^nbits
// amplitudes.
int pass_min_bits(sq_dtype_t dt);
int pass_chunk_bits(sq_dtype_t dt, int nbits);

// Steps of a gate list on an nq-bit state in chunks of 2^cb amplitudes (cb <=
// nq; every step is one gate when cb < pass_min_bits).  masks[g]: the state
// bits gate g acts on (0 for a global phase).  alone: gates have kernels of their
// own, and a gate that no other joins is a step of one gate instead of a pass.
// Gates are reordered only past gates they share no bit with.
void plan_passes(int nq, int cb, sq_dtype_t dt, const std::vector<uint64_t> &masks, bool alone,
                 std::vector<Step> *steps, std::vector<PassPlan> *passes);

// Whether a pass moves less than its gates would on their own kernels, gate g
// changing the fraction touched[g] of the amplitudes.
bool pass_pays(const PassPlan &p, const std::vector<double> &touched);

// Device form of one block: byte offsets in the chunk's LDS image that the
// block's column (group), wave and row (amplitude) index bits stand for; an
// element's offset is the XOR of its bits' entries.
struct PassBlock {
  uint16_t col[5];
  uint16_t wave[4];
  uint16_t row[5];
  uint16_t k;
  uint16_t n16;   // 16-byte units of the block's matrix image
  uint32_t goff;  // its offset in the pass's matrix image, 16-byte units
};

// Geometry of a pass's chunks.
struct PassGeom {
  uint64_t addr[kPassMaxBits];     // address stride (amplitudes) of chunk bit i
  uint64_t lowmask[kPassMaxBits];  // chunk index -> base: insert zero bits here
  int nins;
  int shift;                       // local bits 0..shift-1 are inserted by a shift
};

PassGeom pass_geom(const PassPlan &p);
// The blocks' device descriptors and, per block, the bytes of its matrix.
std::vector<PassBlock> pass_blocks(const PassPlan &p, sq_dtype_t dt, size_t *image_bytes);
// Matrix image of a pass: `matrix(g)` gives gate g's row-major complex128
// matrix and `targets(g)` / `nt(g)` its targets in the reference's order.
struct PassGates {
  const double *matrices;            // all gates' matrices
  const std::vector<size_t> *moffs;  // gate -> offset in matrices (doubles)
  const std::vector<size_t> *toff;   // gate -> offset in targets
  const std::vector<uint32_t> *targets;
  const std::vector<int> *nt;
  int nq;
};
void pass_image(const PassPlan &p, const std::vector<PassBlock> &blocks, sq_dtype_t dt,
                const PassGates &g, char *img);

// One circuit's pass within a launch over many (kernels_cbatch.hip).
struct PassEntry {
  uint64_t psi;       // amplitude offset of the circuit's state
  uint64_t first;     // first workgroup of the entry: one workgroup a chunk
  uint64_t blocks;    // index of its first block descriptor
  uint64_t image;     // byte offset of its matrix image
  int nblocks;
  int initial;        // the state is |0...0>, not read
  PassGeom geom;
};
// Launch `nwg` workgroups over a table of entries of one chunk size; entry[w] is
// workgroup w's entry.
int launch_pass_entries(int cb, sq_dtype_t dt, void *states, const PassEntry *entries,
                        const uint32_t *entry, const PassBlock *blocks, const void *images,
                        uint64_t nwg, hipStream_t stream);
// The launches that takes.
uint64_t pass_entry_launches(uint64_t nwg);

// Launch a pass over nsets states of nelems amplitudes (state y at
// sv + y * nelems, its matrices at image + y * gstride bytes).
int launch_pass(const PassPlan &p, const PassGeom &geom, sq_dtype_t dt, void *sv,
                uint64_t nelems, uint32_t nsets, const PassBlock *blocks, int nblocks,
                const void *image, uint64_t gstride, hipStream_t stream);

}  // namespace sq
