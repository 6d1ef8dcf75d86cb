// pass_plan.cpp -- host side of the multi-gate passes (no device code).
#include "pass_plan.hpp"

#include <algorithm>
#include <array>
#include <cstring>

namespace sq {

// LDS slot of chunk index e: the XOR of slot weights of e's bits.  Weight i
// is 1 << i with the low bits (5 for complex64: 32 8-byte slots span the
// banks; 4 for complex128: 16 16-byte slots) replaced by these values, so
// that the group bits of (nearly) every choice of block targets map onto all
// banks: any 8 of the 13 complex64 values span the 5 low bits in all but 5 of
// the 1287 cases, any 7 of the 12 complex128 values always span the 4.
static const uint32_t kHash64[kPassMaxBits] = {1, 2, 4, 8, 16, 15, 23, 14, 5, 25, 6, 19, 26};
static const uint32_t kHash128[12] = {1, 2, 4, 8, 3, 9, 14, 7, 6, 12, 13, 11};

static uint32_t slot_weight(sq_dtype_t dt, int i) {
  if (dt == SQ_COMPLEX64) return (i < 5 ? 0u : 1u << i) | kHash64[i];
  return (i < 4 ? 0u : 1u << i) | kHash128[i];
}

namespace {

// Next unplaced gate of each bit (position in Planner::perbit).
using Front = std::array<int, 64>;

struct Planner {
  const std::vector<uint64_t> &masks;
  std::vector<std::vector<int>> perbit;  // gates on each bit, program order
  Front ptr;

  bool ready(const Front &p, int g) const {
    for (uint64_t m = masks[g]; m; m &= m - 1) {
      const int b = __builtin_ctzll(m);
      if (perbit[b][p[b]] != g) return false;
    }
    return true;
  }
  int head(const Front &p, int b) const {
    return p[b] < (int)perbit[b].size() ? perbit[b][p[b]] : -1;
  }
  void take(Front &p, int g) const {
    for (uint64_t m = masks[g]; m; m &= m - 1) p[__builtin_ctzll(m)]++;
  }
  // Place every ready gate inside `set`.
  void absorb(Front &p, uint64_t set, std::vector<int> *out) const {
    bool progress = true;
    while (progress) {
      progress = false;
      for (uint64_t m = set; m; m &= m - 1) {
        const int g = head(p, __builtin_ctzll(m));
        if (g < 0 || (masks[g] & ~set) || !ready(p, g)) continue;
        take(p, g);
        out->push_back(g);
        progress = true;
      }
    }
  }
};

}  // namespace

// Blocks of a pass: each gate joins the last block that holds one of its bits
// (or an earlier-made later block) if their union stays within 4 targets or
// inside a block of 5; gates on 5 targets open their own.
static void make_blocks(const std::vector<int> &gates, const std::vector<uint64_t> &masks,
                        uint64_t local, std::vector<PassBlockPlan> *out) {
  struct B {
    uint64_t m;
    std::vector<int> g;
  };
  std::vector<B> bl;
  for (int g : gates) {
    const uint64_t m = masks[g];
    int lo = -1;
    for (int b = (int)bl.size() - 1; b >= 0 && lo < 0; --b)
      if (bl[b].m & m) lo = b;
    int best = -1, grow = 99;
    for (int b = std::max(lo, 0); b < (int)bl.size(); ++b) {
      const uint64_t u = bl[b].m | m;
      const int k = __builtin_popcountll(u);
      if (u != bl[b].m && u != m && k > 4) continue;
      if (k > kMaxK) continue;
      const int gr = k - __builtin_popcountll(bl[b].m);
      if (gr < grow) {
        grow = gr;
        best = b;
      }
    }
    if (best < 0) {
      bl.push_back({m, {g}});
    } else {
      bl[best].m |= m;
      bl[best].g.push_back(g);
    }
  }
  for (auto &b : bl) {
    // at least 4 bits: identity on the lowest local bits not in the block
    for (uint64_t f = local & ~b.m; f && __builtin_popcountll(b.m) < 4; f &= f - 1)
      b.m |= f & -f;
    PassBlockPlan p;
    for (uint64_t m = b.m; m; m &= m - 1) p.bits[p.k++] = __builtin_ctzll(m);
    p.gates = std::move(b.g);
    out->push_back(std::move(p));
  }
}

int pass_min_bits(sq_dtype_t dt) { return dt == SQ_COMPLEX64 ? 10 : 9; }

// Larger chunks hold more gates per pass; these sizes on they still fill the chip
// (layered circuits of depth 10, fused: complex64 19 qubits 129 us with
// 2^13-amplitude chunks and 113 us with 2^12, 20 qubits 122 and 124 us, 22 qubits
// 295 and 356 us; complex128 20 qubits 188 us with 2^12 and 180 us with 2^11, 22
// qubits 563 and 601 us; 64 sets of 20 qubits complex64 7.4 and 8.3 ms).
int pass_chunk_bits(sq_dtype_t dt, int nbits) {
  const int cmax = dt == SQ_COMPLEX64 ? 13 : 12;  // 64 KiB of LDS
  return std::min(nbits, nbits >= (dt == SQ_COMPLEX64 ? 20 : 21) ? cmax : cmax - 1);
}

void plan_passes(int nq, int cb, sq_dtype_t dt, const std::vector<uint64_t> &masks, bool alone,
                 std::vector<Step> *steps, std::vector<PassPlan> *passes) {
  steps->clear();
  passes->clear();
  const int ng = (int)masks.size();
  const bool c64 = dt == SQ_COMPLEX64;
  if (cb < pass_min_bits(dt)) {
    for (int g = 0; g < ng; ++g) steps->push_back({g, -1});
    return;
  }
  const int run = c64 ? 4 : 3;        // 128-byte runs at least
  const uint64_t low = (1ull << run) - 1;
  Planner pl{masks, std::vector<std::vector<int>>(nq), Front{}};
  std::vector<int> phases;
  int left = 0;
  for (int g = 0; g < ng; ++g) {
    if (!masks[g]) {
      phases.push_back(g);  // commutes with everything
      continue;
    }
    ++left;
    for (uint64_t m = masks[g]; m; m &= m - 1) pl.perbit[__builtin_ctzll(m)].push_back(g);
  }
  std::vector<int> t2, btaken;
  while (left) {
    // seed: the earliest ready gate
    int seed = ng;
    for (int b = 0; b < nq; ++b) {
      const int g = pl.head(pl.ptr, b);
      if (g >= 0 && g < seed && pl.ready(pl.ptr, g)) seed = g;
    }
    uint64_t set = low | masks[seed];
    Front ptr = pl.ptr;
    std::vector<int> taken;
    pl.absorb(ptr, set, &taken);
    while (true) {
      // grow by the ready gate that brings the most gates per added bit
      double best = 0.0;
      uint64_t bset = 0;
      Front bptr;
      btaken.clear();
      for (int b = 0; b < nq; ++b) {
        const int g = pl.head(ptr, b);
        if (g < 0 || b != __builtin_ctzll(masks[g]) || !pl.ready(ptr, g)) continue;
        const uint64_t s2 = set | masks[g];
        const int add = __builtin_popcountll(s2) - __builtin_popcountll(set);
        if (__builtin_popcountll(s2) > cb) continue;
        Front p2 = ptr;
        t2.clear();
        pl.absorb(p2, s2, &t2);
        const double score = (double)t2.size() / add;
        if (score > best) {
          best = score;
          bset = s2;
          bptr = p2;
          btaken.swap(t2);
        }
      }
      if (best == 0.0) break;
      set = bset;
      ptr = bptr;
      taken.insert(taken.end(), btaken.begin(), btaken.end());
    }
    if (!alone || taken.size() >= 2) {
      PassPlan p;
      for (int b = 0; b < nq && __builtin_popcountll(set) < cb; ++b) set |= 1ull << b;
      p.local = set;
      p.cb = cb;
      make_blocks(taken, masks, set, &p.blocks);
      p.gates = taken;
      steps->push_back({-1, (int)passes->size()});
      passes->push_back(std::move(p));
    } else {
      steps->push_back({taken[0], -1});
    }
    pl.ptr = ptr;
    left -= (int)taken.size();
  }
  if (passes->empty()) {
    for (int g : phases) steps->push_back({g, -1});
    return;
  }
  // global phases ride in the pass of most gates
  PassPlan &most = *std::max_element(
      passes->begin(), passes->end(),
      [](const PassPlan &a, const PassPlan &b) { return a.gates.size() < b.gates.size(); });
  most.gates.insert(most.gates.end(), phases.begin(), phases.end());
  most.blocks[0].gates.insert(most.blocks[0].gates.end(), phases.begin(), phases.end());
}

bool pass_pays(const PassPlan &p, const std::vector<double> &touched) {
  double sweeps = 0.0;
  for (int g : p.gates) sweeps += touched[g];
  return sweeps > 1.0;
}

PassGeom pass_geom(const PassPlan &p) {
  PassGeom g{};
  int i = 0;
  for (uint64_t m = p.local; m; m &= m - 1) g.addr[i++] = m & -m;
  while ((p.local >> g.shift) & 1) ++g.shift;
  for (uint64_t m = p.local >> g.shift; m; m &= m - 1) g.lowmask[g.nins++] = (m & -m) - 1;
  return g;
}

std::vector<PassBlock> pass_blocks(const PassPlan &p, sq_dtype_t dt, size_t *image_bytes) {
  const bool c64 = dt == SQ_COMPLEX64;
  const int ncol = c64 ? 5 : 4;
  const uint32_t item = c64 ? 8 : 16, banks = c64 ? 31 : 15;
  std::vector<PassBlock> out;
  size_t off = 0;
  for (const PassBlockPlan &b : p.blocks) {
    PassBlock d{};
    int chunk_bit[64];
    int n = 0;
    for (uint64_t m = p.local; m; m &= m - 1) chunk_bit[__builtin_ctzll(m)] = n++;
    uint64_t used = 0;
    for (int j = 0; j < b.k; ++j) {
      const int i = chunk_bit[b.bits[j]];
      used |= 1ull << i;
      d.row[j] = (uint16_t)(slot_weight(dt, i) * item);
    }
    // group bits: the lowest bits whose bank images are independent (no two
    // groups of a row in one bank), topped up if there are not enough
    uint32_t basis[5];
    int nb = 0, nc = 0;
    for (int i = 0; i < p.cb && nc < ncol; ++i) {
      if ((used >> i) & 1) continue;
      uint32_t v = slot_weight(dt, i) & banks;
      for (int q = 0; q < nb; ++q) v = std::min(v, v ^ basis[q]);
      if (!v) continue;
      basis[nb++] = v;
      d.col[nc++] = (uint16_t)(slot_weight(dt, i) * item);
      used |= 1ull << i;
    }
    int nw = 0;
    for (int i = 0; i < p.cb; ++i) {
      if ((used >> i) & 1) continue;
      const uint16_t w = (uint16_t)(slot_weight(dt, i) * item);
      if (nc < ncol) d.col[nc++] = w; else d.wave[nw++] = w;
    }
    d.k = (uint16_t)b.k;
    const size_t bytes = b.k == 5 ? (c64 ? 12288 : 16384) : (c64 ? 6144 : 8192);
    d.n16 = (uint16_t)(bytes / 16);
    d.goff = (uint32_t)(off / 16);
    off += bytes;
    out.push_back(d);
  }
  *image_bytes = off;
  return out;
}

// The block's complex128 matrix (local index bit j = bits[j]), row-major, real
// and imaginary parts apart.
struct BlockMatrix {
  alignas(64) double re[32 * 32], im[32 * 32];
};

static void block_matrix(const PassBlockPlan &b, const PassGates &pg, BlockMatrix *M) {
  const int d = 1 << b.k;
  bool first = true;
  alignas(64) double xr[32 * 32], xi[32 * 32];
  for (int g : b.gates) {
    const double *m = pg.matrices + (*pg.moffs)[g];
    const int k = (*pg.nt)[g], dk = 1 << k;
    // local offset of the gate's index r (reference order: targets[0] the MSB)
    int off[1 << kMaxK] = {0}, mask = 0;
    for (int t = 0; t < k; ++t) {
      const int bit = pg.nq - 1 - (int)(*pg.targets)[(*pg.toff)[g] + t];
      int j = 0;
      while (b.bits[j] != bit) ++j;
      mask |= 1 << j;
      for (int r = 0; r < dk; ++r)
        if ((r >> (k - 1 - t)) & 1) off[r] |= 1 << j;
    }
    if (first) {  // the gate itself, the identity on the other bits
      first = false;
      std::fill(M->re, M->re + d * d, 0.0);
      std::fill(M->im, M->im + d * d, 0.0);
      for (int base = 0; base < d; ++base) {
        if (base & mask) continue;
        for (int r = 0; r < dk; ++r)
          for (int s = 0; s < dk; ++s) {
            M->re[(base | off[r]) * d + (base | off[s])] = m[2 * (r * dk + s)];
            M->im[(base | off[r]) * d + (base | off[s])] = m[2 * (r * dk + s) + 1];
          }
      }
      continue;
    }
    bool diag = true;
    for (int r = 0; r < dk && diag; ++r)
      for (int s = 0; s < dk && diag; ++s)
        diag = r == s || (m[2 * (r * dk + s)] == 0.0 && m[2 * (r * dk + s) + 1] == 0.0);
    if (diag) {
      for (int base = 0; base < d; ++base) {
        if (base & mask) continue;
        for (int r = 0; r < dk; ++r) {
          const double mr = m[2 * (r * dk + r)], mi = m[2 * (r * dk + r) + 1];
          double *yr = M->re + (base | off[r]) * d, *yi = M->im + (base | off[r]) * d;
          for (int c = 0; c < d; ++c) {
            const double a = yr[c];
            yr[c] = mr * a - mi * yi[c];
            yi[c] = mr * yi[c] + mi * a;
          }
        }
      }
      continue;
    }
    if (k == 1) {  // row pairs in place
      const double a0 = m[0], b0 = m[1], a1 = m[2], b1 = m[3];
      const double a2 = m[4], b2 = m[5], a3 = m[6], b3 = m[7];
      const bool real = b0 == 0.0 && b1 == 0.0 && b2 == 0.0 && b3 == 0.0;
      for (int base = 0; base < d; ++base) {
        if (base & mask) continue;
        double *__restrict__ r0 = M->re + base * d, *__restrict__ i0 = M->im + base * d;
        double *__restrict__ r1 = M->re + (base | mask) * d, *__restrict__ i1 = M->im + (base | mask) * d;
        if (real) {
          for (int c = 0; c < d; ++c) {
            const double x0 = r0[c], y0 = i0[c], x1 = r1[c], y1 = i1[c];
            r0[c] = a0 * x0 + a1 * x1;
            i0[c] = a0 * y0 + a1 * y1;
            r1[c] = a2 * x0 + a3 * x1;
            i1[c] = a2 * y0 + a3 * y1;
          }
          continue;
        }
        for (int c = 0; c < d; ++c) {
          const double x0 = r0[c], y0 = i0[c], x1 = r1[c], y1 = i1[c];
          r0[c] = (a0 * x0 - b0 * y0) + (a1 * x1 - b1 * y1);
          i0[c] = (a0 * y0 + b0 * x0) + (a1 * y1 + b1 * x1);
          r1[c] = (a2 * x0 - b2 * y0) + (a3 * x1 - b3 * y1);
          i1[c] = (a2 * y0 + b2 * x0) + (a3 * y1 + b3 * x1);
        }
      }
      continue;
    }
    for (int base = 0; base < d; ++base) {
      if (base & mask) continue;
      for (int s = 0; s < dk; ++s) {
        std::memcpy(xr + s * d, M->re + (base | off[s]) * d, d * sizeof(double));
        std::memcpy(xi + s * d, M->im + (base | off[s]) * d, d * sizeof(double));
      }
      for (int r = 0; r < dk; ++r) {
        double *yr = M->re + (base | off[r]) * d, *yi = M->im + (base | off[r]) * d;
        for (int c = 0; c < d; ++c) yr[c] = yi[c] = 0.0;
        for (int s = 0; s < dk; ++s) {
          const double mr = m[2 * (r * dk + s)], mi = m[2 * (r * dk + s) + 1];
          if (mr == 0.0 && mi == 0.0) continue;
          const double *ar = xr + s * d, *ai = xi + s * d;
          for (int c = 0; c < d; ++c) {
            yr[c] += mr * ar[c] - mi * ai[c];
            yi[c] += mr * ai[c] + mi * ar[c];
          }
        }
      }
    }
  }
}

// Three bf16 parts of each of the n (at most 1024) values v, each part a nearest
// 8-bit value to what the ones before leave: t - (t - v) with t = (2^45 + 1) v
// keeps a double's 8 leading bits (Veltkamp), which a float then holds exactly.
// v is used up.
static void split_bf16(double *__restrict__ v, int n, uint16_t *p0, uint16_t *p1, uint16_t *p2) {
  float f[1024];
  for (uint16_t *out : {p0, p1, p2}) {
    for (int i = 0; i < n; ++i) {
      const double t = v[i] * (0x1p45 + 1.0);
      f[i] = (float)(t - (t - v[i]));
      v[i] -= f[i];
    }
    for (int i = 0; i < n; ++i) {
      uint32_t w;
      std::memcpy(&w, f + i, 4);
      out[i] = (uint16_t)(w >> 16);
    }
  }
}

void pass_image(const PassPlan &p, const std::vector<PassBlock> &blocks, sq_dtype_t dt,
                const PassGates &pg, char *img) {
  const bool c64 = dt == SQ_COMPLEX64;
  BlockMatrix M;
  for (size_t i = 0; i < blocks.size(); ++i) {
    const PassBlockPlan &b = p.blocks[i];
    block_matrix(b, pg, &M);
    const int d = 1 << b.k;
    char *dst = img + (size_t)blocks[i].goff * 16;
    if (c64) {
      // bf16 fragments (kernels_pass.hip): 5 targets the real and imaginary
      // matrices, 4 targets the real 32x32 form, each in three parts of two
      // fragments of 64 lanes x 8 columns
      uint16_t *f = (uint16_t *)dst;
      uint16_t re[3][1024], im[3][1024];
      split_bf16(M.re, d * d, re[0], re[1], re[2]);
      split_bf16(M.im, d * d, im[0], im[1], im[2]);
      // column c = 16t + 8h + j of row r: fragment t, lane r + 32h, entry j
      for (int p3 = 0; p3 < 3; ++p3)
        for (int h8 = 0; h8 < 4; ++h8)
          for (int row = 0; row < 32; ++row) {
            const int at = (h8 >> 1) * 512 + (row + 32 * (h8 & 1)) * 8;
            uint16_t *o = f + p3 * 1024 + at;
            if (b.k == 5) {
              std::memcpy(o, re[p3] + row * 32 + 8 * h8, 16);
              std::memcpy(o + 3 * 1024, im[p3] + row * 32 + 8 * h8, 16);
            } else {  // real form: row 2r + c', columns 2o, 2o + 1
              const uint16_t *er = re[p3] + (row >> 1) * 16 + 4 * h8;
              const uint16_t *ei = im[p3] + (row >> 1) * 16 + 4 * h8;
              for (int q = 0; q < 4; ++q) {
                o[2 * q] = (row & 1) ? ei[q] : er[q];
                o[2 * q + 1] = (row & 1) ? er[q] : (uint16_t)(ei[q] ^ 0x8000u);
              }
            }
          }
      continue;
    }
    double *f = (double *)dst;
    for (int o = 0; o < d; ++o)
      for (int r = 0; r < d; ++r) {
        const double re = M.re[r * d + o], im = M.im[r * d + o];
        if (b.k == 5) {  // entry (o, r): {Re, Im}
          f[2 * (o * d + r)] = re;
          f[2 * (o * d + r) + 1] = im;
        } else {  // real form: row 2r + c, column 2o + c', column-major
          const int e0 = 2 * o * 32 + 2 * r, e1 = e0 + 32;
          f[e0] = re;
          f[e0 + 1] = im;
          f[e1] = -im;
          f[e1 + 1] = re;
        }
      }
  }
}

}  // namespace sq
