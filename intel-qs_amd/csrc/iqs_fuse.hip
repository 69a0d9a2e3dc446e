// Lists of one- and two-qubit gates applied together (iqsh_apply_gates): planning over the
// gates' dependency graph, and the tile kernel that applies many dense blocks in one pass.
//
// A pass gates the positions of one tile: the lowest ones (so that every row of the tile fills
// cache lines) and 8 or 9 others.  It takes every gate that becomes ready on them,
// grouped into dense blocks of up to four positions; a workgroup loads its tile of 2^M
// amplitudes into registers, applies the blocks one after the other on the matrix cores,
// exchanging the tile through LDS where a block needs other positions in its lanes and
// registers, and stores the tile.  200 random 1- and 2-qubit gates on 32 qubits are 11 passes
// of 3-4 blocks instead of 26 passes of one 5-position block.
//
// What bounds it (complex64, 30 qubits, 120 random gates, 7 passes of 4 blocks): a pass takes 4.5
// ms, of which its loads and stores alone are 3.5 ms (4.9 TB/s of 2S in 128-byte rows) and its
// matrix products alone 2.5 ms (48 products per block and amplitude; the matrix cores are
// busy 0.56 of the time); the phases of the 5 workgroups on a CU overlap in part.  61.3 ms
// as 20 passes of 5-position blocks -> 33.1 ms.  complex128, 29 qubits, 100 gates: 27.7 ms in 6
// passes.  On registers of 20 qubits and below a workgroup per CU runs alone, and a block
// costs about 4 us (exchange and its barriers 2, products 1.3): 10 brick layers of 20 qubits
// 790 -> 141 us with the host's planning (65 us).  Error against 64 bits: complex64, 200 random
// gates on 24 qubits, 7.5e-7 (5-position blocks 8.2e-7: sums of 32 terms instead of 16), with four
// real products instead of three 0.9 of that at 1.1 times the time; complex128, the 20-qubit
// brick, 1.9e-15 (5-position blocks 2.5e-15).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "../../include/iqs_hip.h"
#include "iqs_internal.hpp"
#include "iqs_kernels.hpp"

using namespace iqsk;

namespace {

// ---------------------------------------------------------------------------------------
// Planning

// A D x D gate while others are multiplied into it.  A block's matrix acts alike on every amplitude,
// so the roundings of these products do not average out as those of the amplitudes do, but add up
// to a drift of the norm; they are rounded once, at the end.  Until then an entry is h + l with h a
// multiple of 2^-24: for entries up to 1 products of two h and their sums are exact, and what
// involves an l is small enough that its rounding does not count.  (Entries of any size are as
// good as plain products at least.  The same in long double takes twice as long.)  Error of 60
// brick layers of 12 qubits: 2.1e-15, with plain products 3.0e-15, with every gate multiplied into
// the two-qubit gate by itself 1.7e-14; 10 layers of 20 qubits 1.9e-15 in 141 us, 4.1e-15 by
// itself in as many.  Registers in complex64 take plain products in double, far below their own
// rounding (X false: l is not used).
template <int D, bool X>
struct Wide {
  double h[2][D][D], l[2][D][D];  // real and imaginary parts

  Wide() = default;
  explicit Wide(const double* m)
  {
    for (int r = 0; r < D; ++r)
      for (int c = 0; c < D; ++c)
        for (int p = 0; p < 2; ++p) put(p, r, c, *m++, 0);
  }
  void put(int p, int r, int c, double hi, double lo)
  {
    constexpr double k = 1.5 * (1 << 28);  // sums with k are multiples of 2^-24
    const double v = hi + lo;
    h[p][r][c] = X ? (v + k) - k : hi;
    if (X) l[p][r][c] = (hi - h[p][r][c]) + lo;
  }
  double low(int p, int r, int c) const { return X ? l[p][r][c] : 0.0; }
  Wide operator*(const Wide& y) const
  {
    Wide z;
    for (int r = 0; r < D; ++r) {
      double h0[D] = {}, h1[D] = {}, l0[D] = {}, l1[D] = {};
      for (int k = 0; k < D; ++k) {
        const double a = h[0][r][k], b = h[1][r][k], al = low(0, r, k), bl = low(1, r, k);
        if (a == 0 && b == 0 && al == 0 && bl == 0) continue;
        for (int c = 0; c < D; ++c) {
          const double u = y.h[0][k][c], v = y.h[1][k][c];
          h0[c] += a * u - b * v;
          h1[c] += a * v + b * u;
          if constexpr (X) {
            const double ul = y.l[0][k][c], vl = y.l[1][k][c];
            l0[c] += (a * ul - b * vl) + (al * (u + ul) - bl * (v + vl));
            l1[c] += (a * vl + b * ul) + (al * (v + vl) + bl * (u + ul));
          }
        }
      }
      for (int c = 0; c < D; ++c) {
        z.put(0, r, c, h0[c], l0[c]);
        z.put(1, r, c, h1[c], l1[c]);
      }
    }
    return z;
  }
  void write(double* m) const
  {
    for (int r = 0; r < D; ++r)
      for (int c = 0; c < D; ++c)
        for (int p = 0; p < 2; ++p) *m++ = h[p][r][c] + low(p, r, c);
  }
};

// hi (x) lo: index bit 1 under hi, bit 0 under lo; one of them may be null, for the identity.
template <bool X>
Wide<4, X> kron(const Wide<2, X>* hi, const Wide<2, X>* lo)
{
  Wide<4, X> z;
  if (!hi || !lo) {
    std::memset(&z, 0, sizeof z);
    const Wide<2, X>& x = hi ? *hi : *lo;
    const int s = hi ? 2 : 1, o = 3 - s;  // strides of x's index and of the other
    for (int p = 0; p < 2; ++p)
      for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
          for (int k = 0; k < 2; ++k) {
            z.h[p][i * s + k * o][j * s + k * o] = x.h[p][i][j];
            if (X) z.l[p][i * s + k * o][j * s + k * o] = x.l[p][i][j];
          }
    return z;
  }
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) {
      const double a = hi->h[0][i][j], b = hi->h[1][i][j], al = hi->low(0, i, j), bl = hi->low(1, i, j);
      for (int r = 0; r < 2; ++r)
        for (int c = 0; c < 2; ++c) {
          const double u = lo->h[0][r][c], v = lo->h[1][r][c], ul = lo->low(0, r, c), vl = lo->low(1, r, c);
          z.put(0, 2 * i + r, 2 * j + c, a * u - b * v, (a * ul - b * vl) + (al * (u + ul) - bl * (v + vl)));
          z.put(1, 2 * i + r, 2 * j + c, a * v + b * u, (a * vl + b * ul) + (al * (v + vl) + bl * (u + ul)));
        }
    }
  return z;
}

// The list with the one-qubit gates on a position multiplied together and into the two-qubit
// gate that follows there (after the last one, into that), and consecutive two-qubit gates on the
// same pair multiplied together: a small product each, instead of one with a block's
// matrix.  A brick layer of 20 qubits (H, rotation on every qubit, 9 or 10 CNOTs) becomes its 9
// or 10 two-qubit gates.
template <bool X>
std::vector<iqsh_gate> merge_gates(const iqsh_gate* g, int ngates)
{
  std::vector<iqsh_gate> out;
  // Per position: the last two-qubit gate of the list there, and the one-qubit gates since, with
  // their own place in the list where none is before them (-1: none).  The matrix of a two-qubit
  // gate that is still last on a position is in `pair` at one of its positions, home[gate].
  int last[64], place[64];
  bool some[64] = {};
  const std::unique_ptr<Wide<2, X>[]> lone(new Wide<2, X>[64]);
  const std::unique_ptr<Wide<4, X>[]> pair(new Wide<4, X>[64]);
  std::vector<uint8_t> home;
  std::fill(last, last + 64, -1);
  std::fill(place, place + 64, -1);
  auto add = [&](const iqsh_gate& x) {
    out.emplace_back();
    out.back().np = x.np;
    out.back().p[0] = x.p[0];
    out.back().p[1] = x.p[1];
    home.push_back((uint8_t)x.p[0]);
    return (int)out.size() - 1;
  };
  // The one-qubit gates on q, which go into a two-qubit gate; null if there are none.
  auto take = [&](unsigned q) -> const Wide<2, X>* {
    if (!some[q]) return nullptr;
    if (place[q] >= 0) out[place[q]].np = 0;
    place[q] = -1;
    some[q] = false;
    return &lone[q];
  };
  // Another gate becomes the last one on q.
  auto leave = [&](unsigned q) {
    const int i = last[q];
    if (i < 0) return;
    const unsigned other = out[i].p[out[i].p[0] == q];
    if (last[other] != i) pair[q].write(out[i].m);
    else if (home[i] == q) {
      pair[other] = pair[q];
      home[i] = (uint8_t)other;
    }
  };
  for (int i = 0; i < ngates; ++i) {
    const iqsh_gate& x = g[i];
    const unsigned a = x.p[0], b = x.p[1];
    if (x.np == 1) {
      if (some[a]) lone[a] = Wide<2, X>(x.m) * lone[a];
      else {
        lone[a] = Wide<2, X>(x.m);
        some[a] = true;
        if (last[a] < 0) place[a] = add(x);
      }
      continue;
    }
    Wide<4, X> m(x.m);
    const Wide<2, X>*ma = take(a), *mb = take(b);
    if (ma || mb) m = m * kron(ma, mb);
    if (last[a] >= 0 && last[a] == last[b]) {
      if (out[last[a]].p[0] != a)  // the same pair the other way round: exchange the index bits
        for (auto* e : {m.h, m.l})
          for (int p = 0; p < 2 && (X || e == m.h); ++p) {
            for (int v = 0; v < 4; ++v) std::swap(e[p][1][v], e[p][2][v]);
            for (int v = 0; v < 4; ++v) std::swap(e[p][v][1], e[p][v][2]);
          }
      Wide<4, X>& z = pair[home[last[a]]];
      z = m * z;
      continue;
    }
    leave(a);
    leave(b);
    last[a] = last[b] = add(x);
    pair[a] = m;
  }
  for (unsigned q = 0; q < 64; ++q) {
    if (last[q] < 0) {
      if (some[q]) lone[q].write(out[place[q]].m);
      continue;
    }
    iqsh_gate& x = out[last[q]];
    if (home[last[q]] != q) continue;
    const bool first = x.p[0] == q;
    const unsigned other = x.p[first];
    const Wide<2, X>*mq = take(q), *mo = last[other] == last[q] ? take(other) : nullptr;
    if (mq || mo) pair[q] = kron(first ? mq : mo, first ? mo : mq) * pair[q];
    pair[q].write(x.m);
  }
  out.erase(std::remove_if(out.begin(), out.end(), [](const iqsh_gate& x) { return x.np == 0; }), out.end());
  return out;
}

// Gates that depend on each other only through the positions they share: gate i is ready when
// the previous gate on each of its positions has been taken.
struct Dag {
  struct Node {
    int next[2];  // following gate on each position, -1 if none
    int npred;
  };
  std::vector<Node> node;
  std::vector<int> ready;  // ascending

  // The gates list[0..count) of `g` (list null: all of them, in order).
  void build(const iqsh_gate* g, const int* list, int count)
  {
    node.assign(count, Node{{-1, -1}, 0});
    int last[64];
    std::fill(last, last + 64, -1);
    for (int i = 0; i < count; ++i) {
      const iqsh_gate& x = g[list ? list[i] : i];
      for (unsigned j = 0; j < x.np; ++j) {
        const int l = last[x.p[j]];
        if (l >= 0) {
          Node& p = node[l];
          if (p.next[0] != i && p.next[1] != i) {
            p.next[p.next[0] >= 0] = i;
            ++node[i].npred;
          }
        }
        last[x.p[j]] = i;
      }
    }
    ready.clear();
    for (int i = 0; i < count; ++i)
      if (!node[i].npred) ready.push_back(i);
  }
  void take(size_t r)
  {
    const Node x = node[ready[r]];
    ready.erase(ready.begin() + (long)r);
    for (int s : x.next)
      if (s >= 0 && --node[s].npred == 0) ready.insert(std::lower_bound(ready.begin(), ready.end(), s), s);
  }
  static uint64_t mask(const iqsh_gate& x)
  {
    return (uint64_t(1) << x.p[0]) | (x.np == 2 ? uint64_t(1) << x.p[1] : 0);
  }
  // How many gates become ready and lie inside `set`, one after the other (nothing is taken).
  unsigned reach(const iqsh_gate* g, const int* list, uint64_t set)
  {
    walk.clear();
    for (int r : ready)
      if (!(mask(g[list ? list[r] : r]) & ~set)) walk.push_back(r);
    for (size_t i = 0; i < walk.size(); ++i)
      for (int s : node[walk[i]].next)
        if (s >= 0) {
          touched.push_back(s);
          if (--node[s].npred == 0 && !(mask(g[list ? list[s] : s]) & ~set)) walk.push_back(s);
        }
    for (int s : touched) ++node[s].npred;
    touched.clear();
    return (unsigned)walk.size();
  }
  // Takes gates into `out` while the positions `set` grow to at most `limit`: all that become
  // ready inside the set, then the set grows by the ready gate that brings the most gates
  // within reach per new position (the oldest of them).  A gate wider than the limit starts a set
  // of its own.  Against growing by the fewest new positions this saves passes and blocks: 200
  // random gates on 32 qubits 11 passes of 38 blocks instead of 13 of 40, 8 brick layers of 28
  // qubits 7 of 36 instead of 11 of 43.
  void absorb(const iqsh_gate* g, const int* list, uint64_t& set, unsigned limit, std::vector<int>& out)
  {
    for (;;) {
      for (size_t r = 0; r < ready.size();) {
        const int i = list ? list[ready[r]] : ready[r];
        if (mask(g[i]) & ~set) {
          ++r;
          continue;
        }
        out.push_back(i);
        take(r);
        r = 0;
      }
      uint64_t best = 0;
      unsigned best_gain = 0, best_add = 1;
      for (int r : ready) {
        const uint64_t m = mask(g[list ? list[r] : r]) & ~set;
        const unsigned add = (unsigned)__builtin_popcountll(m);
        if (set && (unsigned)__builtin_popcountll(set) + add > limit) continue;
        const unsigned gain = reach(g, list, set | m);
        if (gain * best_add > best_gain * add) {
          best = m;
          best_gain = gain;
          best_add = add;
        }
      }
      if (!best) return;
      set |= best;
    }
  }

 private:
  std::vector<int> walk, touched;
};

// The product of a block's gates as a dense 2^k x 2^k matrix; row bit j <-> position pos[j].
struct Product {
  unsigned k = 0;
  unsigned pos[5];
  double re[32][32], im[32][32];

  // One more position: this (x) I, the new index bit above the others.
  unsigned bit_of(unsigned p)
  {
    for (unsigned j = 0; j < k; ++j)
      if (pos[j] == p) return j;
    const unsigned D = 1u << k;
    for (unsigned r = 0; r < D; ++r) {
      std::memcpy(re[r + D] + D, re[r], D * sizeof(double));
      std::memcpy(im[r + D] + D, im[r], D * sizeof(double));
      for (unsigned c = 0; c < D; ++c) re[r + D][c] = im[r + D][c] = re[r][c + D] = im[r][c + D] = 0;
    }
    pos[k] = p;
    return k++;
  }

  // The gates in order, on positions as they come up, then `fill` up to kmin positions.
  void build(const iqsh_gate* g, const std::vector<int>& gates, unsigned kmin, const unsigned* fill)
  {
    k = 0;
    re[0][0] = 1;
    im[0][0] = 0;
    for (int i : gates) {
      const iqsh_gate& x = g[i];
      // Rows of a group differ in the gate's bits only; gate index 2 b(p[0]) + b(p[1]).
      const unsigned d = 1u << x.np;
      const unsigned bit0 = 1u << bit_of(x.p[0]), bit1 = x.np == 2 ? 1u << bit_of(x.p[1]) : 0;
      const unsigned D = 1u << k;
      for (unsigned r = 0; r < D; ++r) {
        if (r & (bit0 | bit1)) continue;
        unsigned row[4];
        for (unsigned t = 0; t < d; ++t)
          row[t] = x.np == 1 ? r | (t ? bit0 : 0) : r | ((t & 2) ? bit0 : 0) | ((t & 1) ? bit1 : 0);
        double nr[4][32], ni[4][32];
        for (unsigned t = 0; t < d; ++t) {
          for (unsigned c = 0; c < D; ++c) nr[t][c] = ni[t][c] = 0;
          for (unsigned s = 0; s < d; ++s) {
            const double ur = x.m[2 * (t * d + s)], ui = x.m[2 * (t * d + s) + 1];
            if (ur == 0 && ui == 0) continue;
            const double *sr = re[row[s]], *si = im[row[s]];
            for (unsigned c = 0; c < D; ++c) {
              nr[t][c] += ur * sr[c] - ui * si[c];
              ni[t][c] += ur * si[c] + ui * sr[c];
            }
          }
        }
        for (unsigned t = 0; t < d; ++t) {
          std::memcpy(re[row[t]], nr[t], D * sizeof(double));
          std::memcpy(im[row[t]], ni[t], D * sizeof(double));
        }
      }
    }
    while (k < kmin) (void)bit_of(*fill++);
  }
};

// ---------------------------------------------------------------------------------------
// The tile kernel

constexpr int kThreadBits = 8;  // most thread bits of a workgroup (256 threads)
// Real matrices of a block: Ur, Ui and Ur + Ui, for the complex product in three real ones.
constexpr int kMats = 3;

// A tile: 2^M amplitudes, 16 per thread: M = 12, or 10 for registers smaller than that.
// complex64 with 2^13 amplitudes in 512 threads: fewer passes on some lists, but two workgroups
// per CU overlap less (30 qubits 43.8 against 38.6 ms with 2^12).  2^10 and 2^11 on registers of
// 13 to 16 qubits were up to 12% faster, from 18 qubits on slower (20 qubits 202 against 205 and
// 230 us).
template <typename T, int M_>
struct FTile {
  static constexpr int M = M_, NB = M - 4, NT = 1 << NB;
  static_assert(NB >= 6 && NB <= kThreadBits, "1..8 wavefronts");
  // The positions every tile holds: rows of at least 128 bytes, whole cache lines.  (complex128
  // with 256-byte rows: 100 random gates on 29 qubits in 7 passes, 31.4 ms, against 6 passes, 28.9.)
  static constexpr int kLowBits = sizeof(T) == 8 ? 3 : 4;
  // Bank of an LDS slot: its low kFold bits (128 bytes).  Slots are tile indices with the
  // higher bits folded into those by XOR, so that tile bit i moves the bank by bit i mod kFold.
  static constexpr int kFold = sizeof(T) == 8 ? 4 : 5;
  static constexpr size_t kFragBytes = sizeof(T) * kMats * 4 * 64;
  static uint16_t slot(unsigned bit) { return (uint16_t)((1u << bit) ^ ((int)bit >= kFold ? 1u << (bit % kFold) : 0)); }
};

// Where a layout keeps the tile bits: thread bit i (lane bits 0-5, then wave bits) and register
// bit j of each thread, as LDS slot contributions.
struct FLayout {
  uint16_t t[kThreadBits];
  uint16_t r[4];
};
// One block: its layout, and whether the tile has to be exchanged into it.
struct FBlock {
  FLayout at;
  uint32_t exchange;
  uint32_t pad;
};
static_assert(sizeof(FBlock) == 32, "block descriptor");

// A pass: the tile's positions, the layout as loaded and as stored (positions of its thread
// and register bits), and the blocks.
struct FPass {
  uint8_t p[16];  // tile positions, ascending
  uint8_t load_t[kThreadBits], load_r[4], store_t[kThreadBits], store_r[4];
  uint16_t exchange_out;
  FLayout load, store;
  unsigned nblocks;
};

// LDS slot part of this thread's index bits.
template <int NB>
__device__ __forceinline__ uint32_t thread_slot(const FLayout& l)
{
  uint32_t s = 0;
#pragma unroll
  for (int i = 0; i < NB; ++i) s ^= ((threadIdx.x >> i) & 1) ? (uint32_t)l.t[i] : 0u;
  return s;
}

__device__ __forceinline__ uint32_t reg_slot(const FLayout& l, int k)
{
  return ((k & 1) ? l.r[0] : 0) ^ ((k & 2) ? l.r[1] : 0) ^ ((k & 4) ? l.r[2] : 0) ^ ((k & 8) ? l.r[3] : 0);
}

// The block on the thread's 16 amplitudes.  Matrix index bits 0, 1 (complex64: 2, 3) are lane
// bits 4, 5, the other two are register bits 0, 1; register bits 2, 3 and the other lanes and
// waves are columns.  Operands of v_mfma_*_16x16x4: A lane l <-> A[l%16][l/16], B lane l <->
// B[l/16][l%16], accumulator element i of lane l <-> D[(l/16)+4i][l%16] (f64) or
// D[4(l/16)+i][l%16] (f32): with A's columns ordered as above, results come out in the
// layout of the inputs.
template <typename T>
__device__ __forceinline__ void block16(T (&xr)[16], T (&xi)[16], const T (&a)[3][4])
{
  using Acc = typename MfmaAcc<T>::t;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    Acc d1{0, 0, 0, 0}, d2{0, 0, 0, 0}, d3{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const T br = xr[4 * q + j], bi = xi[4 * q + j];
      d1 = mfma16x16x4(a[0][j], br, d1);
      d2 = mfma16x16x4(a[1][j], bi, d2);
      d3 = mfma16x16x4(a[2][j], br + bi, d3);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      xr[4 * q + i] = d1[i] - d2[i];
      xi[4 * q + i] = d3[i] - d1[i] - d2[i];
    }
    // Three independent products keep the matrix cores busy; more tiles at once only spill.
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <typename T, int M, bool NT>
__global__ __launch_bounds__((FTile<T, M>::NT), (sizeof(T) == 8 ? 3 : 4)) void k_tile_blocks(
    typename Vec<T>::t* __restrict__ st, FPass ps, const FBlock* __restrict__ blocks, const T* __restrict__ frags)
{
  using F = FTile<T, M>;
  using V = typename Vec<T>::t;
  constexpr int NB = F::NB;
  __shared__ T lds[1 << M];
  const uint64_t G = grid_blocks();
  uint64_t base = (G & 7) ? block_id() : xcd_block(block_id(), G);
#pragma unroll
  for (int i = 0; i < M; ++i) base = ins0(base, ps.p[i]);
  T xr[16], xi[16];
  {
    uint64_t at = base;
#pragma unroll
    for (int i = 0; i < NB; ++i) at |= (uint64_t)((threadIdx.x >> i) & 1) << ps.load_t[i];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      uint64_t o = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if ((k >> j) & 1) o |= uint64_t(1) << ps.load_r[j];
      const V v = ldx<NT>(&st[at + o]);
      xr[k] = v.x;
      xi[k] = v.y;
    }
  }
  FLayout cur = ps.load;
  // Real parts, then imaginary parts through one buffer of 2^M reals: half the LDS of a
  // complex buffer, so that more workgroups share a CU.
  auto exchange = [&](const FLayout& to) {
    const uint32_t from_t = thread_slot<NB>(cur), to_t = thread_slot<NB>(to);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) lds[from_t ^ reg_slot(cur, k)] = xr[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) xr[k] = lds[to_t ^ reg_slot(to, k)];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) lds[from_t ^ reg_slot(cur, k)] = xi[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) xi[k] = lds[to_t ^ reg_slot(to, k)];
    cur = to;
  };
  // Each block's matrix is loaded (from the L2s) while the block before it is multiplied.
  const T* fr = frags + (threadIdx.x & 63);
  auto fetch = [&](T (&a)[kMats][4], unsigned b) {
#pragma unroll
    for (int m = 0; m < kMats; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) a[m][j] = fr[((b * kMats + m) * 4 + j) * 64];
  };
  T a[kMats][4];
  fetch(a, 0);
  FBlock blk = blocks[0];
  for (unsigned b = 0; b < ps.nblocks; ++b) {
    if (blk.exchange) exchange(blk.at);
    const unsigned nb = b + 1 < ps.nblocks ? b + 1 : b;
    T an[kMats][4];
    fetch(an, nb);
    blk = blocks[nb];
    block16(xr, xi, a);
#pragma unroll
    for (int m = 0; m < kMats; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) a[m][j] = an[m][j];
  }
  if (ps.exchange_out) exchange(ps.store);
  {
    uint64_t at = base;
#pragma unroll
    for (int i = 0; i < NB; ++i) at |= (uint64_t)((threadIdx.x >> i) & 1) << ps.store_t[i];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      uint64_t o = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if ((k >> j) & 1) o |= uint64_t(1) << ps.store_r[j];
      V v;
      v.x = xr[k];
      v.y = xi[k];
      stx<NT>(v, &st[at + o]);
    }
  }
}

// ---------------------------------------------------------------------------------------
// Block descriptors and matrices on their way to the device: a ring of kSlots pinned slots
// and their device copies, reused when the pass that reads one has finished.  Calls take
// turns on it (a lock held until a call's last pass is submitted).
constexpr int kSlots = 4;
constexpr unsigned kSlotBlocks = 64;  // blocks of one launch at most
constexpr size_t kSlotBytes = kSlotBlocks * (sizeof(FBlock) + 3 * 4 * 64 * sizeof(double));
struct FuseRing {
  char *host = nullptr, *dev = nullptr;
  hipEvent_t done[kSlots];
  bool used[kSlots] = {};
  int next = 0;
};
FuseRing g_fr;
std::mutex g_fm;

int ring_slot(int* slot)
{
  if (!g_fr.dev) {
    if (!g_fr.host) IQSI_TRY(hipHostMalloc((void**)&g_fr.host, kSlotBytes * kSlots, hipHostMallocDefault));
    for (int i = 0; i < kSlots; ++i) IQSI_TRY(hipEventCreateWithFlags(&g_fr.done[i], hipEventDisableTiming));
    IQSI_TRY(hipMalloc((void**)&g_fr.dev, kSlotBytes * kSlots));
  }
  *slot = g_fr.next;
  g_fr.next = (g_fr.next + 1) % kSlots;
  if (g_fr.used[*slot]) IQSI_TRY(hipEventSynchronize(g_fr.done[*slot]));
  return IQSH_OK;
}

// A layout as tile bits: thread bit i holds tile bit t[i], register bit j tile bit r[j].
struct Bits {
  uint8_t t[kThreadBits], r[4];
};

template <typename T, int M>
FLayout slots_of(const Bits& b)
{
  using F = FTile<T, M>;
  FLayout l{};
  for (int i = 0; i < F::NB; ++i) l.t[i] = F::slot(b.t[i]);
  for (int j = 0; j < 4; ++j) l.r[j] = F::slot(b.r[j]);
  return l;
}

// Lanes on the lowest tile bits, registers on the highest: as loaded and stored.
template <typename T, int M>
Bits plain_layout()
{
  using F = FTile<T, M>;
  Bits b{};
  for (int i = 0; i < F::NB; ++i) b.t[i] = (uint8_t)i;
  for (int j = 0; j < 4; ++j) b.r[j] = (uint8_t)(F::NB + j);
  return b;
}

// The layout of a block on tile bits blk[0..3] (index bits 0, 1 on lane bits 4, 5, index bits 2, 3
// on register bits 0, 1).  Lane bits 0-3 take the lowest four tile bits when they are free (whole
// rows: loaded and stored as they are), else bits that fall on different banks.
template <typename T, int M>
Bits block_layout(const unsigned* blk, bool* rows)
{
  using F = FTile<T, M>;
  uint32_t left = (1u << M) - 1;
  for (int j = 0; j < 4; ++j) left &= ~(1u << blk[j]);
  Bits b{};
  b.t[4] = (uint8_t)blk[0];
  b.t[5] = (uint8_t)blk[1];
  b.r[0] = (uint8_t)blk[2];
  b.r[1] = (uint8_t)blk[3];
  *rows = (left & 15) == 15;
  uint32_t banks = 0;
  for (int i = 0; i < 4; ++i) {
    int pick = -1;
    for (int t = 0; t < M && pick < 0; ++t)
      if (((left >> t) & 1) && !((banks >> (t % F::kFold)) & 1)) pick = t;
    if (pick < 0) pick = __builtin_ctz(left);
    banks |= 1u << (pick % F::kFold);
    left &= ~(1u << pick);
    b.t[i] = (uint8_t)pick;
  }
  for (int i = 6; i < F::NB; ++i) {
    b.t[i] = (uint8_t)__builtin_ctz(left);
    left &= left - 1;
  }
  for (int j = 2; j < 4; ++j) {
    b.r[j] = (uint8_t)__builtin_ctz(left);
    left &= left - 1;
  }
  return b;
}

// The block's real matrices in operand order: frag[m][j][lane] = A_m[lane % 16][column of
// k-step j and lane group lane / 16].
template <typename T>
void write_frags(const Product& u, T* out)
{
  for (int a = 0; a < 16; ++a) {
    // index bits of the matrix: lane part (c) | register part (j) << 2
    const int row = sizeof(T) == 8 ? a : (a >> 2) | ((a & 3) << 2);
    const double *ur = u.re[row], *ui = u.im[row];
    for (int j = 0; j < 4; ++j)
      for (int c = 0; c < 4; ++c) {
        const T r = (T)ur[c | (j << 2)], i = (T)ui[c | (j << 2)];
        T* o = out + j * 64 + c * 16 + a;
        o[0] = r;
        o[4 * 64] = i;
        o[8 * 64] = r + i;
      }
  }
}

struct Planned {
  std::vector<int> gates;
  uint64_t set;
};

// One launch's worth of a pass: its tile and where its blocks begin in the slot.
struct Staged {
  FPass pass;
  unsigned first;
};

// Writes blocks [first, first + count) of a pass on the tile `set` into slot memory at block
// index `at`.
template <typename T, int M>
int stage_pass(const iqsh_gate* g, const std::vector<Planned>& blocks, size_t first, size_t count, uint64_t set, char* host,
               unsigned at, Staged* out)
{
  using F = FTile<T, M>;
  FPass& ps = out->pass;
  ps = FPass{};
  out->first = at;
  unsigned tile_of[64] = {};
  int m = 0;
  for (unsigned p = 0; p < 64; ++p)
    if ((set >> p) & 1) {
      if (m == M) return iqsi::fail(IQSH_ERR_ARG, "more than %d positions in a tile", M);
      tile_of[p] = (unsigned)m;
      ps.p[m++] = (uint8_t)p;
    }
  if (m != M) return iqsi::fail(IQSH_ERR_ARG, "tile of %d positions (%d expected)", m, M);
  FBlock* desc = (FBlock*)host + at;
  T* frag = (T*)(host + kSlotBlocks * sizeof(FBlock)) + (size_t)at * kMats * 4 * 64;
  const Bits plain = plain_layout<T, M>();
  Bits load = plain, last{};
  bool rows = false;
  Product u;
  for (size_t i = 0; i < count; ++i) {
    const Planned& b = blocks[first + i];
    // Its positions, filled up to four with others of the tile (U (x) I).
    unsigned fill[4], tb[4], nf = 0;
    for (int t = M - 1; t >= 0 && nf < 4; --t)
      if (!((b.set >> ps.p[t]) & 1)) fill[nf++] = ps.p[t];
    u.build(g, b.gates, 4, fill);
    for (int j = 0; j < 4; ++j) tb[j] = tile_of[u.pos[j]];
    last = block_layout<T, M>(tb, &rows);
    desc[i].at = slots_of<T, M>(last);
    desc[i].exchange = 1;
    if (i == 0 && rows) {  // loaded in its own layout
      load = last;
      desc[i].exchange = 0;
    }
    write_frags<T>(u, frag + i * kMats * 4 * 64);
  }
  const Bits store = rows ? last : plain;
  for (int i = 0; i < F::NB; ++i) {
    ps.load_t[i] = ps.p[load.t[i]];
    ps.store_t[i] = ps.p[store.t[i]];
  }
  for (int j = 0; j < 4; ++j) {
    ps.load_r[j] = ps.p[load.r[j]];
    ps.store_r[j] = ps.p[store.r[j]];
  }
  ps.load = slots_of<T, M>(load);
  ps.store = slots_of<T, M>(store);
  ps.exchange_out = !rows;
  ps.nblocks = (unsigned)count;
  return IQSH_OK;
}

// Copies the staged blocks to the device and launches their passes.
template <typename T, int M>
int submit(iqsh_handle h, int slot, const std::vector<Staged>& staged, unsigned nblocks)
{
  using F = FTile<T, M>;
  using V = typename Vec<T>::t;
  if (staged.empty()) return IQSH_OK;
  char *host = g_fr.host + slot * kSlotBytes, *dev = g_fr.dev + slot * kSlotBytes;
  IQSI_TRY(hipMemcpyAsync(dev, host, kSlotBlocks * sizeof(FBlock) + nblocks * F::kFragBytes, hipMemcpyHostToDevice,
                          iqsi::stream()));
  const uint64_t G = uint64_t(1) << (h->n - M);
  const dim3 grid((unsigned)std::min<uint64_t>(G, 65536), (unsigned)((G + 65535) / 65536), 1);
  for (const Staged& p : staged) {
    const FBlock* desc = (const FBlock*)dev + p.first;
    const T* frag = (const T*)(dev + kSlotBlocks * sizeof(FBlock)) + (size_t)p.first * kMats * 4 * 64;
    if (iqsi::cached_pass(h, h->size() * h->esz()))
      k_tile_blocks<T, M, false><<<grid, F::NT, 0, iqsi::stream()>>>((V*)h->d, p.pass, desc, frag);
    else
      k_tile_blocks<T, M, true><<<grid, F::NT, 0, iqsi::stream()>>>((V*)h->d, p.pass, desc, frag);
    IQSI_TRY(hipGetLastError());
  }
  IQSI_TRY(hipEventRecord(g_fr.done[slot], iqsi::stream()));
  g_fr.used[slot] = true;
  return IQSH_OK;
}

// A block by itself, one pass: the 2x2 and 4x4 kernels, or that of up to five positions.
int launch_dense(iqsh_handle h, const iqsh_gate* g, const Planned& b)
{
  Product u;
  u.build(g, b.gates, 0, nullptr);
  const unsigned D = 1u << u.k;
  double m[2 * 32 * 32];
  for (unsigned r = 0; r < D; ++r)
    for (unsigned c = 0; c < D; ++c) {
      m[2 * (r * D + c)] = u.re[r][c];
      m[2 * (r * D + c) + 1] = u.im[r][c];
    }
  if (u.k == 1) return iqsh_apply_1q(h, u.pos[0], m);
  if (u.k == 2) return iqsh_apply_2q(h, u.pos[1], u.pos[0], m);
  return iqsh_apply_kq(h, u.k, u.pos, m);
}

// Passes of tile blocks.  Passes are staged until a launch's share of a slot is full, then
// copied and launched together (one copy for a short list; a long one is planned while the
// GPU works on what came before).
constexpr unsigned kSubmitBlocks = 32;

// Whether the gates of a pass are faster as `dense` passes of one 5-position block each than as one
// pass of `tiled` blocks: few positions under many gates (a circuit on five qubits is one such
// block).  From 64 MiB of amplitudes on, where the kernels' time counts, not the host's, a tile's
// block takes about a quarter of a pass of the 5-position kernel in complex128, a fifth in complex64.
// One dense block against 2, 3, 4, 5 and 10 of a tile: complex128, 27 qubits, 885 us against
// 853, 1023, 1244, 1469 and 2646, 22 qubits 37 against 41, 57, 66, 72 and 115; complex64, 27
// qubits, 450 (positions above 5; 635 on the lowest) against 430, 525, 676, 805 and 1387.  Below,
// 21 qubits complex128, 34-79 (planning) against 26-74.
template <typename T>
bool dense_is_faster(iqsh_handle h, size_t tiled, size_t dense)
{
  return h->size() * h->esz() >= (uint64_t(64) << 20) && tiled + 1 >= (sizeof(T) == 8 ? 4 : 5) * dense;
}

template <typename T, int M>
int apply_tiled(iqsh_handle h, const iqsh_gate* g, int ngates, unsigned block, uint64_t* launched)
{
  std::lock_guard<std::mutex> lk(g_fm);
  Dag all, in;
  all.build(g, nullptr, ngates);
  const uint64_t every = (uint64_t(1) << h->n) - 1;
  const uint64_t low = (uint64_t(1) << FTile<T, M>::kLowBits) - 1;
  std::vector<int> gates;
  std::vector<Planned> blocks, dense;
  std::vector<Staged> staged;
  unsigned used = 0;
  int slot = -1;
  auto flush = [&]() -> int {
    const int rc = slot < 0 ? IQSH_OK : submit<T, M>(h, slot, staged, used);
    staged.clear();
    used = 0;
    slot = -1;
    return rc;
  };
  while (!all.ready.empty()) {
    uint64_t set = h->n == (unsigned)M ? every : low;
    gates.clear();
    all.absorb(g, nullptr, set, M, gates);
    // Fill the tile up with the lowest other positions (longer rows).
    for (uint64_t rest = every & ~set; __builtin_popcountll(set) < M; rest &= rest - 1) set |= rest & -rest;
    auto plan = [&](unsigned limit, std::vector<Planned>& list) {
      list.clear();
      in.build(g, gates.data(), (int)gates.size());
      while (!in.ready.empty()) {
        list.push_back(Planned{{}, 0});
        in.absorb(g, gates.data(), list.back().set, limit, list.back().gates);
      }
    };
    plan(std::min(block, 4u), blocks);
    bool alone = blocks.size() == 1 && __builtin_popcountll(blocks[0].set) <= 2;
    if (block == 5) {  // 5-position blocks need at least one pass per five positions
      uint64_t touched = 0;
      for (const Planned& b : blocks) touched |= b.set;
      if (dense_is_faster<T>(h, blocks.size(), (__builtin_popcountll(touched) + 4) / 5)) {
        plan(5, dense);
        if (dense_is_faster<T>(h, blocks.size(), dense.size())) {
          blocks.swap(dense);
          alone = true;
        }
      }
    }
    if (alone) {
      if (int rc = flush()) return rc;
      for (const Planned& b : blocks) {
        if (int rc = launch_dense(h, g, b)) return rc;
        ++*launched;
      }
      continue;
    }
    for (size_t i = 0; i < blocks.size();) {
      if (slot < 0)
        if (int rc = ring_slot(&slot)) return rc;
      const size_t count = std::min<size_t>(kSlotBlocks - used, blocks.size() - i);
      staged.emplace_back();
      if (int rc = stage_pass<T, M>(g, blocks, i, count, set, g_fr.host + slot * kSlotBytes, used, &staged.back())) return rc;
      ++*launched;
      used += (unsigned)count;
      i += count;
      if (used >= kSubmitBlocks)
        if (int rc = flush()) return rc;
    }
  }
  return flush();
}

// One dense block of up to `block` positions per pass: registers smaller than a tile, block kernels
// that the caller has chosen instead of the tiles' three real products, and captures.
int apply_blocks(iqsh_handle h, const iqsh_gate* g, int ngates, unsigned block, uint64_t* launched)
{
  Dag all;
  all.build(g, nullptr, ngates);
  while (!all.ready.empty()) {
    Planned b{{}, 0};
    all.absorb(g, nullptr, b.set, block, b.gates);
    if (int rc = launch_dense(h, g, b)) return rc;
    ++*launched;
  }
  return IQSH_OK;
}

}  // namespace

extern "C" int iqsh_apply_gates(iqsh_handle h, uint64_t ngates, const iqsh_gate* gates, unsigned block, uint64_t* launched)
{
  if (!h || !h->d) return iqsi::fail(IQSH_ERR_ARG, "null or released state handle");
  if (ngates && !gates) return iqsi::fail(IQSH_ERR_ARG, "null gate list");
  if (ngates > 0x7fffffff) return iqsi::fail(IQSH_ERR_NOTSUP, "more than 2^31 gates in one list");
  if (block < 1 || block > 5) return iqsi::fail(IQSH_ERR_ARG, "block size %u out of range", block);
  for (uint64_t i = 0; i < ngates; ++i) {
    const iqsh_gate& x = gates[i];
    if (x.np < 1 || x.np > 2) return iqsi::fail(IQSH_ERR_ARG, "gate %llu on %u positions", (unsigned long long)i, x.np);
    for (unsigned j = 0; j < x.np; ++j)
      if (x.p[j] >= h->n) return iqsi::fail(IQSH_ERR_ARG, "position %u out of range for %u qubits", x.p[j], h->n);
    if (x.np == 2 && x.p[0] == x.p[1]) return iqsi::fail(IQSH_ERR_ARG, "gate positions coincide");
  }
  if (ngates == 1) {
    const iqsh_gate& x = gates[0];
    const int rc = x.np == 1 ? iqsh_apply_1q(h, x.p[0], x.m) : iqsh_apply_2q(h, x.p[0], x.p[1], x.m);
    if (launched) *launched = rc == IQSH_OK;
    return rc;
  }
  uint64_t count = 0;
  int rc;
  // A graph is replayed after the ring's slots have been used again: in a capture every gate is in
  // its kernel's arguments.
  const bool capture = iqsi::capturing();
  if (capture) block = std::min(block, 2u);
  try {
    const std::vector<iqsh_gate> merged =
        h->dtype == IQSH_C128 ? merge_gates<true>(gates, (int)ngates) : merge_gates<false>(gates, (int)ngates);
    gates = merged.data();
    const int ng = (int)merged.size();
    if (h->n < 10 || capture || iqsi::block_kernel() != 1) rc = apply_blocks(h, gates, ng, block, &count);
    else if (h->dtype == IQSH_C128)
      rc = h->n < 12 ? apply_tiled<double, 10>(h, gates, ng, block, &count) : apply_tiled<double, 12>(h, gates, ng, block, &count);
    else
      rc = h->n < 12 ? apply_tiled<float, 10>(h, gates, ng, block, &count) : apply_tiled<float, 12>(h, gates, ng, block, &count);
  } catch (const std::exception& e) {
    return iqsi::fail(IQSH_ERR_ALLOC, "planning %llu gates: %s", (unsigned long long)ngates, e.what());
  }
  if (launched) *launched = count;
  return rc;
}
