// Where the particle kernels put their grid contributions (J_r, J_phi, J_z
// and the bunch rho, all FP64).
//
// GlobalSink: bounds-checked hardware FP64 atomics straight to HBM (used by
// the split entry points and for the charge of bunches).
//
// TileSinkT: three levels, for particles walked by one lane in runs of the same
// cell:
//   1. registers: the contributions of the current cell (ic, kc) to its
//      J_phi / rho corners (ic..ic+1, kc..kc+1), J_z nodes (ic..ic+1, kc) and
//      J_r nodes (ic, kc..kc+1) are summed in FP64 registers and flushed only
//      when the lane moves to a particle in another cell;
//   2. an LDS box of nodes around the block's cells (tile_anchor, tall_init,
//      bunch_init), filled with LDS FP64 atomics;
//   3. nodes outside the box go to GlobalSink.
// After the block the box is added to HBM once (one atomic per touched node).
// Small tiles, of one or two particles per lane, and the bunches whose lanes hold
// one leave out the first level, the FP64 kernels altogether.
#pragma once

#include "context.hpp"

namespace pdp3 {

enum SinkComp { kCR = 0, kCPhi = 1, kCZ = 2, kCRho = 3 };

// j: J_r of the context's grid, with J_phi and J_z the next nr*nz arrays
// (one base pointer instead of three keeps the particle kernels' scalar
// registers from spilling); rho: the bunch charge density, or a caller's array
struct GlobalSink {
  int nr, nz;
  double *j, *rho;
  int *err;
  __device__ __forceinline__ double *base(int comp) const {
    return comp == kCRho ? rho : j + (size_t)comp * ((size_t)nr * (size_t)nz);
  }
  __device__ __forceinline__ void put(int comp, int i, int k, double v) const {
    if ((unsigned)i < (unsigned)nr && (unsigned)k < (unsigned)nz)
      unsafeAtomicAdd(base(comp) + (size_t)i * (size_t)nz + (size_t)k, v);
    else
      atomicOr(err, kErrDomain);
  }
  // a pair of nodes: (i, k), (i+1, k) for J_z; (i, k), (i, k+1) for J_r
  template <int C>
  __device__ __forceinline__ void add2(int i, int k, double v0, double v1) {
    put(C, i, k, v0);
    if (C == kCZ)
      put(C, i + 1, k, v1);
    else
      put(C, i, k + 1, v1);
  }
  // the four corners (i..i+1, k..k+1) of J_phi / rho
  template <int C>
  __device__ __forceinline__ void add4(int i, int k, double v00, double v10, double v01, double v11) {
    put(C, i, k, v00);
    put(C, i + 1, k, v10);
    put(C, i, k + 1, v01);
    put(C, i + 1, k + 1, v11);
  }
  __device__ __forceinline__ void begin_cell(int, int) {}
  __device__ __forceinline__ void flush() {}
};

// BR x BK nodes per component; the plasma box spans 4 rows (i0-1 .. i0+2) by
// 128 columns (a sorted block covers a run of cells along one row).  A bunch
// block is a thin disc of particles injected in the same step: its box has
// BR x BK nodes in 16, 32 or 64 rows (bunch_init)
// ACC: the first level; without it (lanes that hold one particle) every
// contribution goes to the box at once: 8 LDS atomics where the registers'
// stencil takes 12, and no setting up of the registers
template <bool RHO, int BR = 4, int BK = 128, bool ACC = true>
struct TileSinkT {
  static constexpr bool kBunch = RHO;
  static constexpr int kComps = RHO ? 4 : 3;  // rho only where it is deposited
  static constexpr int kR = BR, kK = BK, kSize = kComps * BR * BK;
  GlobalSink g;
  double *box;  // LDS, kComps x kR x kK
  int bi, bk;   // node coordinates of box[.][0][0]
  int bw;       // columns of the box in use (a multiple of the wavefront or kK)
  int shift;    // bunches: log2 of the box's columns
  int ic, kc;   // cell of the register accumulator
  // scalar accumulators (no arrays: a runtime index would push them to scratch)
  double p00, p10, p01, p11;  // J_phi corners (ic+di, kc+dk)
  double r00, r10, r01, r11;  // rho corners (bunches only)
  double z0, z1;              // J_z at (ic, kc), (ic+1, kc)
  double x0, x1;              // J_r at (ic, kc), (ic, kc+1)

  // a node past the box.  (A bunch's zeros, such as the J_phi of one without v_phi,
  // a third of its atomics, are left out, as flush leaves them out.)
  __device__ __forceinline__ void past_put(int comp, int i, int k, double v) {
    if (ACC || !RHO || v != 0.0) g.put(comp, i, k, v);
  }
  __device__ __forceinline__ int rows() const { return RHO ? (BR * BK) >> shift : BR; }
  __device__ __forceinline__ int stride() const { return RHO ? 1 << shift : BK; }
  __device__ __forceinline__ double *at(int li, int lk) const { return box + (RHO ? li << shift : li * BK) + lk; }
  // whole stencils at once: one bounds check and atomics at fixed offsets; the
  // nodes of one that leaves the box go to HBM, in a loop (one copy of put)
  template <int C>
  __device__ __forceinline__ void box_put2(int i, int k, double v0, double v1) {
    const int li = i - bi, lk = k - bk;
    if ((unsigned)li < (unsigned)(rows() - (C == kCZ)) && (unsigned)lk < (unsigned)(bw - (C != kCZ))) {
      double *q = at(li, lk) + C * BR * BK;
      atomicAdd(q, v0);
      atomicAdd(q + (C == kCZ ? stride() : 1), v1);
      return;
    }
#pragma nounroll
    for (int n = 0; n < 2; n++) past_put(C, i + (C == kCZ ? n : 0), k + (C == kCZ ? 0 : n), n ? v1 : v0);
  }
  template <int C>
  __device__ __forceinline__ void box_put4(int i, int k, double v00, double v10, double v01, double v11) {
    const int li = i - bi, lk = k - bk;
    if ((unsigned)li < (unsigned)(rows() - 1) && (unsigned)lk < (unsigned)(bw - 1)) {
      double *q = at(li, lk) + C * BR * BK;
      atomicAdd(q, v00);
      atomicAdd(q + stride(), v10);
      atomicAdd(q + 1, v01);
      atomicAdd(q + stride() + 1, v11);
      return;
    }
#pragma nounroll
    for (int n = 0; n < 4; n++)
      past_put(C, i + (n & 1), k + (n >> 1), n < 2 ? (n ? v10 : v00) : (n == 2 ? v01 : v11));
  }
  // whole stencils: straight into the accumulators when they are centred on
  // the accumulator's cell (the common case: no select chains), else the box
  template <int C>
  __device__ __forceinline__ void add2(int i, int k, double v0, double v1) {
    if (ACC && i == ic && k == kc) {
      if (C == kCZ) {
        z0 += v0;
        z1 += v1;
      } else {
        x0 += v0;
        x1 += v1;
      }
      return;
    }
    box_put2<C>(i, k, v0, v1);
  }
  template <int C>
  __device__ __forceinline__ void add4(int i, int k, double v00, double v10, double v01, double v11) {
    if (ACC && i == ic && k == kc && (C == kCPhi || RHO)) {
      if (C == kCPhi) {
        p00 += v00; p10 += v10; p01 += v01; p11 += v11;
      } else {
        r00 += v00; r10 += v10; r01 += v01; r11 += v11;
      }
      return;
    }
    box_put4<C>(i, k, v00, v10, v01, v11);
  }
  __device__ __forceinline__ void put_nz(int comp, int i, int k, double v) {
    if (v != 0.0) g.put(comp, i, k, v);
  }
  // the accumulators' stencil (nodes ic..ic+1, kc..kc+1) in one piece: when
  // it lies inside the box, one bounds check and LDS atomics at fixed offsets
  // from one address (zeros included: cheaper than testing each value);
  // otherwise node by node to HBM
  __device__ __forceinline__ void flush() {
    if (!ACC || ic < 0) return;
    const int li = ic - bi, lk = kc - bk;
    if ((unsigned)li < (unsigned)(rows() - 1) && (unsigned)lk < (unsigned)(bw - 1)) {
      double *q = at(li, lk);
      constexpr int C = BR * BK;
      const int BS = stride();
      atomicAdd(q + kCPhi * C, p00);
      atomicAdd(q + kCPhi * C + BS, p10);
      atomicAdd(q + kCPhi * C + 1, p01);
      atomicAdd(q + kCPhi * C + BS + 1, p11);
      if (RHO) {
        atomicAdd(q + kCRho * C, r00);
        atomicAdd(q + kCRho * C + BS, r10);
        atomicAdd(q + kCRho * C + 1, r01);
        atomicAdd(q + kCRho * C + BS + 1, r11);
      }
      atomicAdd(q + kCZ * C, z0);
      atomicAdd(q + kCZ * C + BS, z1);
      atomicAdd(q + kCR * C, x0);
      atomicAdd(q + kCR * C + 1, x1);
    } else {
      put_nz(kCPhi, ic, kc, p00);
      put_nz(kCPhi, ic + 1, kc, p10);
      put_nz(kCPhi, ic, kc + 1, p01);
      put_nz(kCPhi, ic + 1, kc + 1, p11);
      if (RHO) {
        put_nz(kCRho, ic, kc, r00);
        put_nz(kCRho, ic + 1, kc, r10);
        put_nz(kCRho, ic, kc + 1, r01);
        put_nz(kCRho, ic + 1, kc + 1, r11);
      }
      put_nz(kCZ, ic, kc, z0);
      put_nz(kCZ, ic + 1, kc, z1);
      put_nz(kCR, ic, kc, x0);
      put_nz(kCR, ic, kc + 1, x1);
    }
    p00 = p10 = p01 = p11 = 0.0;
    r00 = r10 = r01 = r11 = 0.0;
    z0 = z1 = x0 = x1 = 0.0;
  }
  // the next particle's contributions are centred on cell (i, k)
  __device__ __forceinline__ void begin_cell(int i, int k) {
    if (ACC && (i != ic || k != kc)) {
      flush();
      ic = i;
      kc = k;
    }
  }
};
using TileSink = TileSinkT<false>;  // plasma species: no rho
using BunchSink = TileSinkT<true, 16, 32>;
using TileSinkTall = TileSinkT<false, 8, 128, false>;  // small tiles: see tall_init
using BunchSinkOne = TileSinkT<true, 16, 32, false>;

// One grid's node deposits of a tile (charge weighting outside the loop, the
// density probe): the four corners of the lane's current cell in registers, an
// LDS box of kR x kK nodes, the grid.
struct NodeSink {
  static constexpr int kR = 4, kK = 128, kSize = kR * kK;
  GlobalSink g;
  double *out;  // the grid
  double *box;  // LDS
  int bi, bk, ic, kc;
  double r00, r10, r01, r11;

  __device__ __forceinline__ void init(const GlobalSink &gs, double *grid, double *lds, int ai, int ak) {
    g = gs;
    out = grid;
    box = lds;
    bi = ai - 1;
    bk = ak - 2;
    ic = kc = -1;
    r00 = r10 = r01 = r11 = 0.0;
    for (int t = threadIdx.x; t < kSize; t += blockDim.x) box[t] = 0.0;
  }
  __device__ __forceinline__ void grid_put(int i, int k, double v) {
    if ((unsigned)i < (unsigned)g.nr && (unsigned)k < (unsigned)g.nz)
      unsafeAtomicAdd(out + (size_t)i * (size_t)g.nz + (size_t)k, v);
    else
      atomicOr(g.err, kErrDomain);
  }
  __device__ __forceinline__ void put(int i, int k, double v) {
    const int li = i - bi, lk = k - bk;
    if ((unsigned)li < (unsigned)kR && (unsigned)lk < (unsigned)kK)
      atomicAdd(box + li * kK + lk, v);
    else
      grid_put(i, k, v);
  }
  template <int C>
  __device__ __forceinline__ void add4(int i, int k, double v00, double v10, double v01, double v11) {
    if (i == ic && k == kc) {
      r00 += v00; r10 += v10; r01 += v01; r11 += v11;
      return;
    }
    put(i, k, v00);
    put(i + 1, k, v10);
    put(i, k + 1, v01);
    put(i + 1, k + 1, v11);
  }
  __device__ __forceinline__ void flush() {
    if (ic < 0) return;
    put(ic, kc, r00);
    put(ic + 1, kc, r10);
    put(ic, kc + 1, r01);
    put(ic + 1, kc + 1, r11);
    r00 = r10 = r01 = r11 = 0.0;
  }
  __device__ __forceinline__ void begin_cell(int i, int k) {
    if (i != ic || k != kc) {
      flush();
      ic = i;
      kc = k;
    }
  }
  __device__ __forceinline__ void to_grid() {  // after flush and __syncthreads
    for (int t = threadIdx.x; t < kSize; t += blockDim.x)
      if (box[t] != 0.0) grid_put(bi + t / kK, bk + t % kK, box[t]);
  }
};

// The anchor cell of a tile of cell-sorted particles, from the cells (i, k)
// of its logical particles 0, 16 and 32 (live: a living particle; uniform
// values, so that the choice runs on the scalar unit): the median row of the
// living samples (the smaller when two live) and the smallest column among
// the samples in that row; (0, 0) when none lives.  Between sorts a few
// particles have moved to a neighbouring cell; a box anchored at one of them
// that moved to another row would serve the tile's own row only at its edge,
// so one such stray among the three samples is outvoted.  A sample one
// column off is harmless: the boxes keep two columns below the anchor.
__device__ __forceinline__ void tile_anchor(const bool (&live)[3], const int (&i)[3], const int (&k)[3], int &ai,
                                            int &ak) {
  constexpr int kNone = 0x7fffffff;
  int r[3];
#pragma unroll
  for (int j = 0; j < 3; j++) r[j] = live[j] ? i[j] : kNone;
  const int n = (int)live[0] + (int)live[1] + (int)live[2];
  if (n == 0) {
    ai = ak = 0;
    return;
  }
  const int lo = min(min(r[0], r[1]), r[2]);
  ai = lo;
  if (n == 3) ai = r[0] + r[1] + r[2] - lo - max(max(r[0], r[1]), r[2]);  // the median (rows are small)
  int col = kNone;
#pragma unroll
  for (int j = 0; j < 3; j++)
    if (live[j] && i[j] == ai) col = min(col, k[j]);
  ak = col;
}

// block prologue: anchor the box one row and two columns below the given
// cell (the tile's anchor, or a bunch block's smallest cell) and clear its
// first `width` columns (bunch_init has cleared a bunch's)
template <class T>
__device__ __forceinline__ void box_init(double *box, int anchor_i, int anchor_k, int width, T &s,
                                         const GlobalSink &g) {
  if (!T::kBunch) {
    for (int t = threadIdx.x / 64; t < T::kComps * T::kR; t += blockDim.x / 64)
      for (int c = threadIdx.x % 64; c < width; c += 64) box[t * T::kK + c] = 0.0;
  }
  s.g = g;
  s.box = box;
  s.bi = anchor_i - 1;
  s.bk = anchor_k - 2;
  s.bw = width;
  s.ic = -1;
  s.kc = -1;
  s.p00 = s.p10 = s.p01 = s.p11 = 0.0;
  s.r00 = s.r10 = s.r01 = s.r11 = 0.0;
  s.z0 = s.z1 = s.x0 = s.x1 = 0.0;
}

// block epilogue: add the box to the grid (after __syncthreads)
template <class T>
__device__ __forceinline__ void box_flush(const double *box, const T &s) {
  if (T::kBunch) {
    constexpr int kPlane = T::kR * T::kK;
    for (int t = threadIdx.x; t < T::kSize; t += blockDim.x) {
      const double v = box[t];
      if (v == 0.0) continue;
      const int n = t % kPlane;
      s.g.put(t / kPlane, s.bi + (n >> s.shift), s.bk + (n & (s.bw - 1)), v);
    }
    return;
  }
  for (int t = threadIdx.x / 64; t < T::kComps * T::kR; t += blockDim.x / 64)
    for (int c = threadIdx.x % 64; c < s.bw; c += 64) {
      const double v = box[t * T::kK + c];
      if (v == 0.0) continue;
      const int comp = t / T::kR;
      s.g.put(comp, s.bi + t - comp * T::kR, s.bk + c, v);
    }
}

}  // namespace pdp3

namespace pdp3 {
// smallest (i, k) over the block of two per-thread candidates (INT_MAX when
// the thread saw no living particle); every thread gets the result
__device__ __forceinline__ void block_min2(int &i, int &k) {
  __shared__ int mi[8], mk[8];
  for (int off = 32; off > 0; off >>= 1) {
    i = min(i, __shfl_xor(i, off));
    k = min(k, __shfl_xor(k, off));
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    mi[wave] = i;
    mk[wave] = k;
  }
  __syncthreads();
  i = mi[0];
  k = mk[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); w++) {
    i = min(i, mi[w]);
    k = min(k, mk[w]);
  }
}

// block prologue of a bunch: the box lies one row and two columns below the
// smallest cell of the block's living particles, in the shape (16 x 32, 32 x 16,
// 64 x 8 nodes) that covers the most of the cells up to the largest, three rows
// and four columns of it being margins.  (i, k), (i1, k1): the thread's smallest
// and largest cell (INT_MAX, -1: none living); false: none lives in the block.
// Particles past a 16 x 32 box alone made a bunch of 20 rows, in the order of
// injection, a chain of grid atomics: 1e5 and 1e6 particles 185 and 1880 us
// (FP64; 173 and 1957 in FP32), 20 and 94 us (16 and 75) in its own shape; of four
// rows 19 and 94 us as before.  The choice is scalar arithmetic after one barrier.
template <int WAVES, class T>
__device__ __forceinline__ bool bunch_init(double *box, int i, int k, int i1, int k1, T &s, const GlobalSink &g) {
  // the block's extent: minima of i, k, ~i1 and ~k1
  __shared__ int part[4][WAVES];
  int m[4] = {i, k, ~i1, ~k1};
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int j = 0; j < 4; j++) m[j] = min(m[j], __shfl_xor(m[j], off));
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int j = 0; j < 4; j++) part[j][threadIdx.x >> 6] = m[j];
  for (int t = threadIdx.x; t < T::kSize; t += blockDim.x) box[t] = 0.0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; j++) {
#pragma unroll
    for (int w = 0; w < WAVES; w++) m[j] = min(m[j], part[j][w]);
    m[j] = __builtin_amdgcn_readfirstlane(m[j]);
  }
  if (m[0] == 0x7fffffff) return false;
  const int ni = ~m[2] - m[0] + 1, nk = ~m[3] - m[1] + 1;
  constexpr int kNodes = T::kR * T::kK;
  s.shift = 5;
  if (ni > T::kR - 3) {
    int best = 0;
#pragma unroll
    for (int t = 5; t >= 3; t--) {
      const int cells = min(ni, (kNodes >> t) - 3) * min(nk, (1 << t) - 4);
      if (cells > best) {
        best = cells;
        s.shift = t;
      }
    }
  }
  static_assert(T::kBunch && T::kK == 32, "the first shape");
  box_init(box, m[0], m[1], 1 << s.shift, s, g);
  return true;
}

// the cell that a plasma block's boxes are centred on: the median of nine of its
// particles in the order of cells (a few that have drifted off since the species
// was in that order do not move it, as they would the smallest cell); (0, 0)
// where none of the nine lives.  After 2400 steps without a sort 2.6e5 particles
// at 8 per cell took the tangent step 231 us around the smallest cell in four
// rows, 101 us around the median in six (76 and 69 us where they lie in order,
// all with IEEE divisions).
__device__ __forceinline__ void block_median(int &i, int &k, bool live) {
  constexpr int kN = 9, kEvery = 28;
  __shared__ unsigned long long cell[kN], med;
  if (threadIdx.x % kEvery == kEvery / 2 && threadIdx.x < kN * kEvery)
    cell[threadIdx.x / kEvery] = live ? (unsigned long long)i << 32 | (unsigned)k : ~0ull;
  if (threadIdx.x == 0) med = 0;
  __syncthreads();
  if (threadIdx.x < kN) {
    const unsigned me = threadIdx.x;
    const unsigned long long mine = cell[me];
    int less = 0, all = 0;
#pragma unroll
    for (unsigned j = 0; j < kN; j++) {
      const unsigned long long o = cell[j];
      all += o != ~0ull;
      less += o < mine || (o == mine && j < me);
    }
    if (mine != ~0ull && less == all / 2) med = mine;
  }
  __syncthreads();
  i = (int)(med >> 32);
  k = (int)med;
}

// block prologue of a small tile (one or two particles per lane): the box lies
// around the median cell of nine of its particles, four rows and as many
// columns either side, 64 columns where the tile's particles span no more than
// 56 cells of a sorted species of n particles, else 128.  Without sorts particles
// drift off for thousands of steps; with a box of 4 x 128 nodes from the tile's first
// cell the FP64 step of 4e6 particles went from 0.35 to 0.50 ms over 2000 steps
// (200 x 1000 cells), with this one it stays.  (i, k): the thread's cell.
template <class T>
__device__ __forceinline__ void tall_init(double *box, int i, int k, bool live, int particles, long long n, T &s,
                                          const GlobalSink &g) {
  const int width = particles * (long long)(g.nr - 1) * (g.nz - 1) > 56 * n ? T::kK : T::kK / 2;
  box_init(box, 0, 0, width, s, g);
  block_median(i, k, live);  // and the barrier that the cleared box needs
  s.bi = i - (T::kR / 2 - 1);
  s.bk = k - (width / 2 - 1);
}
}  // namespace pdp3
