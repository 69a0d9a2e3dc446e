// Layers of one 2x2 gate on every qubit (U^(x)n), forward and adjoint: kernels and launch.
// Entry points in iqs_layer.hip; one translation unit per precision instantiates do_layer.
//
// A layer runs in tile passes.  A workgroup takes a tile of 2^M amplitudes into registers
// (2^LR per thread), applies the gate to every tile bit that the pass gates, and writes the
// tile back, so one read and one write of the state serve many qubits:
//   * the low pass gates positions 0 .. M-1: a tile is one contiguous run of the state;
//   * a high pass gates m <= M - LR positions p0 .. p0+m-1: the tile holds those and the
//     c = M - m >= LR lowest positions, so every row of it is a run of 2^c amplitudes.
// At 28 qubits a layer is 3 passes (M = 12: 12 + 8 + 8 positions).
//
// Inside a tile the thread's registers hold LR consecutive tile bits, first the top ones (as
// loaded: consecutive threads, consecutive amplitudes), then the others after an exchange
// through LDS; gates are register-local.  The low pass takes two exchanges, a high pass one,
// none if m <= LR.  The last window is bits LR .. 2 LR - 1, where consecutive threads again
// hold runs of 2^LR amplitudes (256 bytes).
//
// What bounds it: HBM (a pass reads and writes the state, or both states, once).  At 28
// qubits complex128 a forward pass runs at 5.76 TB/s (low, with the QAOA phase) and 5.3
// (high: 256-byte rows), an adjoint pass at 5.7 and 5.5, the in-place scale of the state at
// 6.5; the exchanges (one write and one read of LDS per amplitude each) and the products
// are each under a third of that time.  A layer takes 4.73 ms forward and 9.57 ms adjoint
// (7.45 and 18.2 with one lane pass over 8 positions and register passes over 5 and 4 above,
// which moved the state 5 and 6 times); 25 qubits complex64, weighted: 8.45 -> 4.1 ms for
// cost and gradient at p = 4; 14 qubits complex128: 700 -> 200 us at p = 6.
//
// Adjoint: the gates of a layer act on different qubits, so each generator G_q commutes
// with every gate of the layer except its own, and inserting G_q after U_q equals inserting
// it after the whole layer.  Each window therefore takes its qubits' terms
// 2 Im <lam| G_q |psi> on the amplitudes it holds, then applies Uinv to them.  Sums in FP64:
// per-workgroup partials, summed in a fixed order (bitwise reproducible).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "../../include/iqs_hip.h"
#include "iqs_internal.hpp"
#include "iqs_kernels.hpp"

namespace iqsl {

using namespace iqsk;

// Im(conj(y) * (a x0 + b x1)) with the product in FP64.
template <typename V>
__device__ __forceinline__ double im_term(const V& y, const Cx<double>& a, const V& x0, const Cx<double>& b, const V& x1)
{
  const double gr = (a.r * (double)x0.x - a.i * (double)x0.y) + (b.r * (double)x1.x - b.i * (double)x1.y);
  const double gi = (a.r * (double)x0.y + a.i * (double)x0.x) + (b.r * (double)x1.y + b.i * (double)x1.x);
  return (double)y.x * gi - (double)y.y * gr;
}

// Kernel form flags: kFormGX, the generator is X (two products per term instead of ten);
// kFormRX, the 2x2 has a real diagonal and an imaginary off-diagonal (the mixer RX(2 beta)
// and its inverse), so a row of the product is d x_same + i o x_other: four products instead
// of eight.
constexpr int kFormGX = 1, kFormRX = 2;

// Generator term of one amplitude of a pair (x0, x1): Im(conj(y) (G x)_row), row 1 if hi.
template <int F, typename V>
__device__ __forceinline__ double gen_term(const V& y, const Mat2<double>& g, const V& x0, const V& x1, bool hi)
{
  if constexpr ((F & kFormGX) != 0) {
    const V o = hi ? x0 : x1;
    // complex64 mixer: the product in FP32 (of FP32 amplitudes), summed in FP64 by the caller
    if constexpr (sizeof(o.x) == 4 && (F & kFormRX) != 0) return (double)(y.x * o.y - y.y * o.x);
    return (double)y.x * (double)o.y - (double)y.y * (double)o.x;
  }
  return hi ? im_term(y, g.m10, x0, g.m11, x1) : im_term(y, g.m00, x0, g.m01, x1);
}

template <int F, typename T, typename V>
__device__ __forceinline__ V urow(const Mat2<T>& u, const V& x0, const V& x1, bool hi)
{
  if constexpr ((F & kFormRX) != 0) {
    const T d = hi ? u.m11.r : u.m00.r, o = hi ? u.m10.i : u.m01.i;
    const V xs = hi ? x1 : x0, xo = hi ? x0 : x1;
    V r;
    r.x = d * xs.x - o * xo.y;
    r.y = d * xs.y + o * xo.x;
    return r;
  } else {
    return hi ? cmad2(u.m10, x0, u.m11, x1) : cmad2(u.m00, x0, u.m01, x1);
  }
}

// The QAOA phase exp(-i gamma cut(x)) of a low pass, applied while the thread's registers
// hold tile bits (= positions) a .. a+LR-1.  E(x) = XOR of inc[b] over the set bits b of x has
// bit e set if edge e is cut (linear over GF(2)), so E(x) = E(thread's other bits) ^ E(register
// index), the second the same for every thread.
//  * unit weights: cut = popcount E, phase from a table in LDS.
//  * weighted: every edge touches no register bit, one, or two.  cut(r) = base +
//    sum_j side[j][r_j] + both[r], where base sums the cut edges of the first kind, side[j][v]
//    the cut edges at register bit j when it has value v, both[r] (the same for every thread)
//    those between two register bits; the phase is the product of the parts' phases, so a
//    thread takes 2 LR + 1 sincos for its 2^LR amplitudes instead of one each.  Only cut
//    edges are ever added, so weights of very different size do not cancel.
struct CutWin {
  uint64_t none;             // edges that touch no register bit
  uint64_t one[5];           // edges with exactly one end at a register bit, by bit
  double both[32];           // cut of the edges between two register bits, by register index
  double both_re[32], both_im[32];  // its phase
};

constexpr int kCutNone = 0, kCutUnit = 1, kCutWeighted = 2;
struct NoCut {};
template <int CUT> using CutArg = std::conditional_t<CUT == kCutNone, NoCut, CutSpec>;
template <int CUT> using WinArg = std::conditional_t<CUT == kCutWeighted, CutWin, NoCut>;

// Tile of one pass: c, p0 as above (low pass: c = M).
struct TilePass {
  unsigned c, p0;
};

template <typename T, int M_, int LR_>
struct LTile {
  static constexpr int M = M_, LR = LR_, R = 1 << LR, NT = 1 << (M - LR);
  static_assert(M >= 2 * LR && M <= 3 * LR, "three windows of LR bits cover the tile");
  static_assert(NT >= 64 && NT <= 1024, "1..16 wavefronts");
  using V = typename Vec<T>::t;

  // Tile index of register k of thread tid when the registers hold tile bits [a, a + LR).
  static __device__ __forceinline__ uint32_t lidx(uint32_t tid, int k, int a)
  {
    return (tid & ((1u << a) - 1u)) | ((uint32_t)k << a) | ((tid >> a) << (a + LR));
  }
  // LDS slot of a tile index: the low LR bits XOR-ed with the next LR bits, so that the
  // 2^LR consecutive lanes of every window fall on different banks.
  static __device__ __forceinline__ uint32_t phys(uint32_t u) { return u ^ ((u >> LR) & (R - 1u)); }

  // Exchange the window [A, A+LR) for [B, B+LR), real parts then imaginary parts through one
  // buffer of 2^M reals: half the LDS of a complex buffer, which is what lets four
  // workgroups share a CU in the forward passes.  lds is free on entry and in use on exit.
  template <int A, int B>
  static __device__ __forceinline__ void exchange(V (&v)[R], T* lds)
  {
    const uint32_t tid = threadIdx.x;
#pragma unroll
    for (int k = 0; k < R; ++k) lds[phys(lidx(tid, k, A))] = v[k].x;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < R; ++k) v[k].x = lds[phys(lidx(tid, k, B))];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < R; ++k) lds[phys(lidx(tid, k, A))] = v[k].y;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < R; ++k) v[k].y = lds[phys(lidx(tid, k, B))];
  }
};

// Workgroup sum of v (fixed order: lanes by xor-shuffle, then the waves in order) stored at
// *out by thread 0.
template <int NT>
__device__ __forceinline__ void wg_sum_store(double v, double* out)
{
  __shared__ double sh[NT / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0;
    for (int w = 0; w < NT / 64; ++w) s += sh[w];
    *out = s;
  }
  __syncthreads();
}

// The gate on the window's bits j (tile bit a + j) that the pass gates (a + j in [c, end)):
// the generator terms of a bit first (adjoint), then the update of its pairs.
template <typename LT, bool ADJ, int F, typename T>
__device__ __forceinline__ void window_gates(typename LT::V (&x)[LT::R], typename LT::V (&y)[ADJ ? LT::R : 1], int a,
                                             int begin, int end, const Mat2<T>& u, const Mat2<double>& g, double& acc)
{
  using V = typename LT::V;
#pragma unroll
  for (int j = 0; j < LT::LR; ++j) {
    if (a + j < begin || a + j >= end) continue;
#pragma unroll
    for (int k = 0; k < LT::R; ++k) {
      if ((k >> j) & 1) continue;
      const int k1 = k | (1 << j);
      const V p0 = x[k], p1 = x[k1];
      if constexpr (ADJ) {
        const V l0 = y[k], l1 = y[k1];
        acc += gen_term<F>(l0, g, p0, p1, false) + gen_term<F>(l1, g, p0, p1, true);
        y[k] = urow<F>(u, l0, l1, false);
        y[k1] = urow<F>(u, l0, l1, true);
      }
      x[k] = urow<F>(u, p0, p1, false);
      x[k1] = urow<F>(u, p0, p1, true);
    }
    // The sum is taken here: only used at the end of the kernel, it would otherwise be sunk
    // there with every amplitude that its terms need (a thousand spilled registers).
    if constexpr (ADJ) __asm__ volatile("" : "+v"(acc));
  }
}

// The phase on the window at tile bit a of a low pass (see CutWin).  Adjoint: the phase term
// cut Im(conj(lam) psi) into accg before both states are multiplied.
template <typename LT, bool ADJ, int CUT, int A, typename T>
__device__ __forceinline__ void window_phase(typename LT::V (&x)[LT::R], typename LT::V (&y)[ADJ ? LT::R : 1], uint64_t t,
                                             const CutSpec& cs, const WinArg<CUT>& cw, const Cx<T>* ph, double& accg)
{
  constexpr int LR = LT::LR, R = LT::R, M = LT::M;
  uint64_t e = 0;
  for (uint64_t r = t; r; r &= r - 1) e ^= cs.inc.c[M + __builtin_ctzll(r)];
#pragma unroll
  for (int b = 0; b < M - LR; ++b) {
    const uint64_t ib = cs.inc.c[b < A ? b : b + LR];
    e ^= ((threadIdx.x >> b) & 1) ? ib : 0;
  }
  auto use = [&](int k, double cut, const Cx<T>& f) {
    if constexpr (ADJ) {
      accg += cut * ((double)y[k].x * x[k].y - (double)y[k].y * x[k].x);
      y[k] = cmul(f, y[k]);
    }
    x[k] = cmul(f, x[k]);
  };
  if constexpr (CUT == kCutUnit) {
#pragma unroll
    for (int k = 0; k < R; ++k) {
      uint64_t ek = 0;
#pragma unroll
      for (int j = 0; j < LR; ++j)
        if ((k >> j) & 1) ek ^= cs.inc.c[A + j];
      const int ic = __popcll(e ^ ek);
      use(k, (double)ic, ph[ic]);
    }
  } else {
    // Sums over cut edges: no register bit set in e (register index 0).
    double base = 0, side[LR][2];
    Cx<double> fbase, fside[LR][2];
    for (uint64_t m = cw.none; m; m &= m - 1) {
      const int i = __builtin_ctzll(m);
      base += ((e >> i) & 1) ? cs.w[i] : 0.0;
    }
    sincos(cs.gamma * base, &fbase.i, &fbase.r);
    fbase.i = -fbase.i;
#pragma unroll
    for (int j = 0; j < LR; ++j) {
      double s0 = 0, s1 = 0;
      for (uint64_t m = cw.one[j]; m; m &= m - 1) {
        const int i = __builtin_ctzll(m);
        const bool cut = (e >> i) & 1;
        s0 += cut ? cs.w[i] : 0.0;
        s1 += cut ? 0.0 : cs.w[i];
      }
      side[j][0] = s0;
      side[j][1] = s1;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        sincos(cs.gamma * side[j][v], &fside[j][v].i, &fside[j][v].r);
        fside[j][v].i = -fside[j][v].i;
      }
    }
    // Partial sums and products over the register bits from the top down, so that each
    // amplitude adds one bit's part to those it shares with its neighbours.
    double cs_[LR + 1];
    Cx<double> f_[LR + 1];
    cs_[LR] = base;
    f_[LR] = fbase;
#pragma unroll
    for (int k = 0; k < R; ++k) {
#pragma unroll
      for (int j = LR - 1; j >= 0; --j) {
        if ((k & ((1 << j) - 1)) != 0) continue;  // bits >= j unchanged since the last k
        const int v = (k >> j) & 1;
        cs_[j] = cs_[j + 1] + side[j][v];
        f_[j].r = f_[j + 1].r * fside[j][v].r - f_[j + 1].i * fside[j][v].i;
        f_[j].i = f_[j + 1].r * fside[j][v].i + f_[j + 1].i * fside[j][v].r;
      }
      const double br = cw.both_re[k], bi = cw.both_im[k];
      const Cx<T> f{(T)(f_[0].r * br - f_[0].i * bi), (T)(f_[0].r * bi + f_[0].i * br)};
      use(k, cs_[0] + cw.both[k], f);
    }
  }
}

// Waves per SIMD that a pass's registers are held to.  complex128 forward, the upper passes of a
// general 2x2: with four of them 56 of 128 registers were spilled (24 qubits 316 -> 244 us with
// three, 28 qubits 4.80 -> 4.59 ms).  Its adjoint spills 66 with two; one wave is slower (28 qubits
// 12.2 -> 15.4 ms).
template <typename T, int LR, bool ADJ, bool LOW, int F, int CUT>
constexpr int layer_waves()
{
  if (ADJ) return sizeof(T) == 8 ? 2 : 3;
  return CUT == kCutWeighted || LR == 5 || (sizeof(T) == 8 && !LOW && F == 0) ? 3 : 4;
}

// One pass.  LOW: the low pass (c = M), with the QAOA phase (CUT) before the gates going
// forward and after them (undone) in the adjoint.  part (adjoint): the workgroup's sum of
// generator terms at part[block], of phase terms at part[blocks + block].
template <typename T, int M, int LR, bool ADJ, bool LOW, int F, int CUT, bool NT>
__global__ __launch_bounds__((LTile<T, M, LR>::NT), (layer_waves<T, LR, ADJ, LOW, F, CUT>())) void k_layer_tile(
    typename Vec<T>::t* __restrict__ psi, typename Vec<T>::t* __restrict__ lam, TilePass tp, Mat2<T> u, Mat2<double> g,
    CutArg<CUT> cs, WinArg<CUT> cw, double* __restrict__ part)
{
  using LT = LTile<T, M, LR>;
  using V = typename LT::V;
  constexpr int R = LT::R;
  constexpr int TOP = M - LR;  // first window
  __shared__ T lds[1 << M];
  __shared__ Cx<T> ph[CUT == kCutUnit ? 65 : 1];
  const uint32_t tid = threadIdx.x;
  const uint64_t G = grid_blocks();
  const uint64_t t = (G & 7) ? block_id() : xcd_block(block_id(), G);
  const unsigned c = LOW ? M : tp.c;
  // Position map of the tile: bits below c in place, bits c.. at p0..; t fills the rest.
  const unsigned p0 = LOW ? M : tp.p0, mg = M - c;
  const uint64_t base = LOW ? t << M : ((t & ((uint64_t(1) << (p0 - c)) - 1)) << c) | ((t >> (p0 - c)) << (p0 + mg));
  auto gmap = [&](uint32_t i) -> uint64_t {
    return LOW ? (uint64_t)i : (i & ((1u << c) - 1u)) | ((uint64_t)(i >> c) << p0);
  };
  if constexpr (CUT == kCutUnit)
    for (unsigned i = tid; i <= cs.ne && i < 65; i += LT::NT) ph[i] = Cx<T>{(T)cs.ph_re[i], (T)cs.ph_im[i]};
  V x[R], y[ADJ ? R : 1];
  double acc = 0, accg = 0;
  {
    const uint64_t at = base | gmap(LT::lidx(tid, 0, TOP));
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const uint64_t off = gmap((uint32_t)k << TOP);
      x[k] = ldx<NT>(&psi[at + off]);
      if constexpr (ADJ) y[k] = ldx<NT>(&lam[at + off]);
    }
  }
  if (CUT == kCutUnit) __syncthreads();
  if constexpr (!ADJ && CUT != kCutNone) window_phase<LT, ADJ, CUT, TOP>(x, y, t, cs, cw, ph, accg);
  window_gates<LT, ADJ, F>(x, y, TOP, LOW ? 0 : c, M, u, g, acc);
  auto store = [&](auto win) {
    constexpr int A = decltype(win)::value;
    const uint64_t at = base | gmap(LT::lidx(tid, 0, A));
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const uint64_t off = gmap((uint32_t)k << A);
      stx<NT>(x[k], &psi[at + off]);
      if constexpr (ADJ) stx<NT>(y[k], &lam[at + off]);
    }
  };
  if constexpr (LOW) {
    LT::template exchange<TOP, 0>(x, lds);
    if constexpr (ADJ) {
      __syncthreads();
      LT::template exchange<TOP, 0>(y, lds);
    }
    window_gates<LT, ADJ, F>(x, y, 0, 0, LR, u, g, acc);
    __syncthreads();
    LT::template exchange<0, LR>(x, lds);
    if constexpr (ADJ) {
      __syncthreads();
      LT::template exchange<0, LR>(y, lds);
    }
    window_gates<LT, ADJ, F>(x, y, LR, LR, TOP, u, g, acc);
    if constexpr (ADJ && CUT != kCutNone) window_phase<LT, ADJ, CUT, LR>(x, y, t, cs, cw, ph, accg);
    store(std::integral_constant<int, LR>{});
  } else if (c < TOP) {
    LT::template exchange<TOP, LR>(x, lds);
    if constexpr (ADJ) {
      __syncthreads();
      LT::template exchange<TOP, LR>(y, lds);
    }
    window_gates<LT, ADJ, F>(x, y, LR, c, TOP, u, g, acc);
    store(std::integral_constant<int, LR>{});
  } else {
    store(std::integral_constant<int, TOP>{});
  }
  if constexpr (ADJ) {
    wg_sum_store<LT::NT>(acc, part + block_id());
    if (CUT != kCutNone) wg_sum_store<LT::NT>(accg, part + G + block_id());
  }
}

// Sums over workgroups, taken on the way: a pass reserves a run of partials on the device, a
// kernel sums pending runs in a fixed order into pinned host memory when the buffer or its
// argument list is full, and the host waits once, at the end (iqs_layer.hip).
constexpr int kMaxSums = 32;
struct SumRuns {
  uint64_t off[kMaxSums], len[kMaxSums];
};
class LayerSums {
 public:
  // For passes of at most `run` partials in groups of at most `group` runs, `total` runs in all.
  int begin(uint64_t run, int group, uint64_t total);
  // Space for `count` (<= kMaxSums) consecutive runs of `run` partials each; their sums become
  // results [taken(), taken() + count).
  int take(uint64_t run, int count, double** part);
  uint64_t taken() const { return done_ + n_; }
  int flush();
  // Every result, after the stream has been waited for.
  int finish(const double** results);

 private:
  SumRuns runs_;
  uint64_t used_ = 0, done_ = 0;
  int n_ = 0;
};

// One layer's operands.
struct LayerArgs {
  iqsh_handle psi, lam;  // lam: adjoint only
  const double* u;       // 2x2 (adjoint: the inverse)
  const double* g;       // generator (adjoint)
  const CutSpec* cs;     // QAOA phase, or null
  // Adjoint: results of sum_q Im <lam| G_q |psi>, one per pass, then with cs Im <lam| C |psi>.
  LayerSums* sums;
};

// Passes of a layer, and the partials of one.
struct LayerShape {
  unsigned passes;
  uint64_t run;
};

// The window data of a weighted cut when the registers hold positions a .. a+LR-1.
inline void build_cut_window(const CutSpec& cs, unsigned a, unsigned lr, CutWin* cw)
{
  uint64_t once = 0, twice = 0;
  for (unsigned j = 0; j < lr; ++j) {
    twice |= once & cs.inc.c[a + j];
    once |= cs.inc.c[a + j];
  }
  const uint64_t all = cs.ne >= 64 ? ~uint64_t(0) : (uint64_t(1) << cs.ne) - 1;
  cw->none = all & ~once;
  for (unsigned j = 0; j < lr; ++j) cw->one[j] = cs.inc.c[a + j] & ~twice;
  for (unsigned r = 0; r < (1u << lr); ++r) {
    uint64_t e = 0;
    for (unsigned j = 0; j < lr; ++j)
      if ((r >> j) & 1) e ^= cs.inc.c[a + j];
    double s = 0;
    for (uint64_t m = e & twice; m; m &= m - 1) s += cs.w[__builtin_ctzll(m)];
    cw->both[r] = s;
    cw->both_re[r] = std::cos(cs.gamma * s);
    cw->both_im[r] = -std::sin(cs.gamma * s);
  }
}

inline dim3 tile_grid(uint64_t G) { return dim3((unsigned)std::min<uint64_t>(G, 65536), (unsigned)((G + 65535) / 65536), 1); }

template <typename T, int M, int LR, bool ADJ, int F, bool NT = true>
int layer_m(const LayerArgs& a, LayerShape* shape)
{
  using V = typename Vec<T>::t;
  using LT = LTile<T, M, LR>;
  if (a.psi->n < (unsigned)M) return iqsi::fail(IQSH_ERR_NOTSUP, "tile of %d bits in a register of %u qubits", M, a.psi->n);
  const double* um = a.u;
  const Mat2<T> u{{(T)um[0], (T)um[1]}, {(T)um[2], (T)um[3]}, {(T)um[4], (T)um[5]}, {(T)um[6], (T)um[7]}};
  Mat2<double> g{{0, 0}, {0, 0}, {0, 0}, {0, 0}};
  if (ADJ) g = Mat2<double>{{a.g[0], a.g[1]}, {a.g[2], a.g[3]}, {a.g[4], a.g[5]}, {a.g[6], a.g[7]}};
  V* psi = (V*)a.psi->d;
  V* lam = ADJ ? (V*)a.lam->d : nullptr;
  const unsigned n = a.psi->n, rest = n - M, high = (rest + (M - LR) - 1) / (M - LR);
  const uint64_t G = uint64_t(1) << (n - M);
  if (shape) {
    *shape = {high + 1, G};
    return IQSH_OK;
  }
  const dim3 grid = tile_grid(G);
  // Forward: the low pass first (it carries the phase layer, applied before the mixer);
  // adjoint: last (the phase is undone after the whole mixer).
  auto low_pass = [&]() -> int {
    const TilePass tp{M, M};
    double* p = nullptr;
    if (ADJ)  // with a phase its terms follow the generator terms
      if (int rc = a.sums->take(G, a.cs ? 2 : 1, &p)) return rc;
    if (!a.cs) {
      k_layer_tile<T, M, LR, ADJ, true, F, kCutNone, NT><<<grid, LT::NT, 0, iqsi::stream()>>>(psi, lam, tp, u, g, NoCut{}, NoCut{}, p);
    } else if (!a.cs->weighted) {
      k_layer_tile<T, M, LR, ADJ, true, F, kCutUnit, NT><<<grid, LT::NT, 0, iqsi::stream()>>>(psi, lam, tp, u, g, *a.cs, NoCut{}, p);
    } else {
      CutWin cw{};
      build_cut_window(*a.cs, ADJ ? LR : M - LR, LR, &cw);
      k_layer_tile<T, M, LR, ADJ, true, F, kCutWeighted, NT><<<grid, LT::NT, 0, iqsi::stream()>>>(psi, lam, tp, u, g, *a.cs, cw, p);
    }
    return IQSH_OK;
  };
  if (!ADJ)
    if (int rc = low_pass()) return rc;
  // Positions above the low pass in passes of as equal a size as possible.
  for (unsigned i = 0, p = M; i < high; ++i) {
    const unsigned m = rest / high + (i < rest % high ? 1 : 0);
    const TilePass tp{M - m, p};
    double* part = nullptr;
    if (ADJ)
      if (int rc = a.sums->take(G, 1, &part)) return rc;
    k_layer_tile<T, M, LR, ADJ, false, F, kCutNone, NT><<<grid, LT::NT, 0, iqsi::stream()>>>(psi, lam, tp, u, g, NoCut{}, NoCut{}, part);
    p += m;
  }
  if (ADJ)
    if (int rc = low_pass()) return rc;
  IQSI_TRY(hipGetLastError());
  return IQSH_OK;
}

// Tile size: large tiles (long rows, fewest passes) for registers that fill the chip with
// them; below that the smallest tile that takes no more passes, for more workgroups (18
// qubits complex128 takes 14.1 us with 64 tiles of 2^12, 12.6 with 128 of 2^11, but at 20 qubits
// 2^11 needs one pass more: 21.1 against 25.5 us).  complex64 forward: the same, and from 26 qubits
// on 2^13 with 32 amplitudes per thread (256-byte rows as in complex128) where that is one pass
// less (29 qubits 6.22 -> 5.15 ms) or the products are the short ones (28 qubits RX 2.37 -> 2.32 ms;
// with the weighted phase 2.58 against 2.69), and for the one tile of 13 qubits with those (9.1 ->
// 7.9 us; general 2x2 9.2 against 12.1).  Elsewhere 32 amplitudes leave too few waves: general
// 2x2, 12 qubits 12.8 -> 7.0 us with 16, 15 qubits 15.3 -> 10.4, 19 qubits 24.9 -> 16.7, 25 qubits
// with the weighted phase 343 -> 329, RX 303 -> 278.  The adjoint has psi and lambda in registers: 32
// amplitudes of each left two waves per SIMD and spilled (25 qubits weighted low pass 535 against 287
// us).
template <typename T, bool ADJ, int F>
int layer_n(const LayerArgs& a, LayerShape* shape)
{
  const unsigned n = a.psi->n;
  const bool cached = !shape && iqsi::cached_pass(a.psi, a.psi->size() * sizeof(typename Vec<T>::t) * (ADJ ? 2 : 1));
  if constexpr (sizeof(T) == 4 && !ADJ) {
    const bool short_products = (F & kFormRX) != 0 && !(a.cs && a.cs->weighted);
    if ((n >= 26 && (short_products || (n - 13) % 8 == 0)) || (n == 13 && short_products)) return layer_m<T, 13, 5, ADJ, F>(a, shape);
  }
  if (n <= 10 || (n > 12 && n <= 16) || (sizeof(T) == 4 && ADJ && n == 11)) return layer_m<T, 10, 4, ADJ, F>(a, shape);
  if constexpr (sizeof(T) == 8 || !ADJ)
    if (n == 11 || n == 17 || n == 18) return layer_m<T, 11, 4, ADJ, F>(a, shape);
  return cached ? layer_m<T, 12, 4, ADJ, F, false>(a, shape) : layer_m<T, 12, 4, ADJ, F>(a, shape);
}

// With `shape` only that is filled in.  The RX-form kernels when the 2x2 has a real diagonal and an
// imaginary off-diagonal (the QAOA mixer and its inverse) and, in the adjoint, the generator is
// exactly X; the short terms of X also with any other inverse (28 qubits, adjoint: complex128 11.6 ->
// 10.7 ms, complex64 7.9 -> 6.2).
template <typename T>
int do_layer(const LayerArgs& a, LayerShape* shape)
{
  static const double X[8] = {0, 0, 1, 0, 1, 0, 0, 0};
  const bool rx = a.u[1] == 0 && a.u[2] == 0 && a.u[4] == 0 && a.u[7] == 0;
  if (!a.lam) return rx ? layer_n<T, false, kFormRX>(a, shape) : layer_n<T, false, 0>(a, shape);
  const bool gx = std::equal(a.g, a.g + 8, X);
  if (gx) return rx ? layer_n<T, true, kFormGX | kFormRX>(a, shape) : layer_n<T, true, kFormGX>(a, shape);
  return layer_n<T, true, 0>(a, shape);
}

extern template int do_layer<float>(const LayerArgs&, LayerShape*);
extern template int do_layer<double>(const LayerArgs&, LayerShape*);

}  // namespace iqsl
