// FP32 cell-relative form of the per-particle work of one step.
//
// State per particle: packed cell (bit 31 = dead, bits 16..30 = radial cell
// i, bits 0..15 = axial cell k), offsets a, b in (0, 1] with r = (i + a) dr,
// z = (k + b) dz (the reference's half-open cells (i dx, (i+1) dx],
// include/geometry.h:44), momentum per mass u = gamma v (FP32), weight w.
// Storing offsets instead of absolute coordinates keeps every bit of
// resolution however large the grid is; storing u keeps gamma well
// conditioned near c.
//
// Arithmetic: push and deposit in FP32; every formula of the reference is
// rewritten in cell units without catastrophic cancellation (ring-volume
// weights as products (1-a)(2i+a), the segment integrals of
// simple_current_distribution through log1p-type series, the r-z rotation
// through dy^2/(R+X)); the near-axis cell (1/r, the CYL_VOL annulus weights)
// is evaluated in FP64; the grid accumulation is FP64 (hardware FP64
// atomics); fields and the PML stay FP64.
#include <algorithm>
#include <cstring>
#include <vector>

#include <type_traits>

#include "context.hpp"
#include "sink.hpp"

namespace pdp3 {

namespace {

constexpr uint32_t kDead = 0x80000000u;

// a / b, 1/sqrt(x) and sqrt(x) through the hardware instructions (about 1
// ulp each; no denormal arguments reach them here: the Lorentz factors are
// >= 1, the other arguments are O(1) in cell units or exactly 0)
__device__ __forceinline__ float fdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ float frsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

__device__ __forceinline__ int cell_i(uint32_t c) { return (int)((c >> 16) & 0x7FFF); }
__device__ __forceinline__ int cell_k(uint32_t c) { return (int)(c & 0xFFFF); }
__device__ __forceinline__ uint32_t pack(int i, int k) { return ((uint32_t)i << 16) | (uint32_t)k; }

struct F32Args {
  int nr, nz;
  float hr, hz;      // dt / (2 dr), dt / (2 dz): half-step displacement per unit speed, in cells
  float inv_c2;      // 1 / c^2
  float c1;          // q dt / (2 m) of the species (w cancels, src/particles.cpp:1060)
  float bscale;      // Boris: mu0 c1; Vay: mu0 c1 * 2 c1^2 (the reference's Vay scaling, :1187-1210)
  float escale;      // Boris: c1; Vay: 2 c1
  float kz, kr, kp;  // charge/(4 pi dr^2 dt), charge/(2 pi dr dz dt), charge/(4 pi dz dr^2)
  int pusher;
  int is_bunch;
  int want_rho;
  int n;
  // the context's grid: component c (kER, kEPhi, kEZ, kHHR, kHHPhi, kHHZ) at
  // grid + c * nr * nz (one base pointer instead of six keeps the kernels'
  // scalar registers from spilling)
  const double *grid;
  // per radial cell index i, two entries: {1/(2i), 1/(2(i+1)), 1/(2(i+2)),
  // 1/(2(i+3))} and {1/i, 1/(i+1), 1/(i+1/2), i(i+1)} (1/0 read as 0)
  const float4 *rows;
  int *err;
  uint32_t *cell;
  float *fa, *fb, *ur, *uphi, *uz;
  const float *w;
};

// component c of the grid
__device__ __forceinline__ const double *field(const F32Args &p, int c) {
  return p.grid + (size_t)c * ((size_t)p.nr * (size_t)p.nz);
}

// the element at byte offset `off` from p: a 32-bit offset from a
// uniform base is one VGPR and scalar-base addressing, where an element index
// would be widened to a 64-bit address per array
template <class T>
__device__ __forceinline__ T &at(T *p, unsigned off) {
  return *reinterpret_cast<T *>(reinterpret_cast<char *>(p) + off);
}
template <class T>
__device__ __forceinline__ const T &at(const T *p, unsigned off) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + off);
}

// radial weights of the four-node gathers (src/eField.cpp:204-316,
// src/hField.cpp:159-267) in cell units.  "lo" family (E_r, H_z, H_phi):
// staggered index from r - dr/2; otherwise (E_phi, E_z, H_r) the particle's
// own cell with the CYL_VOL volume on the axis cell.  Weights A (node i_r),
// B (node i_r+1), exactly the reference's ring volume / cell volume ratios
// (which do not sum to one).
struct RadW {
  int ir;
  float A, B;
};
// both radial weight pairs of a particle in cell i at offset a; t is the
// first table entry of row i.  The lo family's denominators 2(l+1), 2(l+3)
// (l = its staggered index, i or i-1) and the own family's 2i, 2(i+2) are all
// entries of that row.
__device__ __forceinline__ void rad_weights(int i, float a, const float4 &t, RadW &lo, RadW &own) {
  // staggered index from r - dr/2: i-1 with offset a+1/2 when a <= 1/2, except
  // on the axis cell, where the reference clamps the index at 0 and keeps the
  // offset a-1/2
  const bool down = a <= 0.5f && i > 0;
  const int ir = down ? i - 1 : i;
  const float al = down ? a + 0.5f : a - 0.5f;
  const float fl = (float)ir, fi = (float)i;
  lo.ir = ir;
  lo.A = (1.f - al) * (2.f * fl + 1.f + al) * (down ? t.x : t.y);
  lo.B = al * (2.f * fl + 2.f + al) * (down ? t.z : t.w);
  own.ir = i;
  if (i == 0) {
    double ad = a;  // axis cell in FP64: CYL_VOL annulus weight
    own.A = (float)((1.0 - ad) * ad * 4.0);
    own.B = (float)(ad * (1.0 + ad) / 4.0);
  } else {
    own.A = (1.f - a) * (2.f * fi + a) * t.x;
    own.B = a * (2.f * fi + 1.f + a) * t.z;
  }
}
struct AxW {
  int kz;
  float b;  // weight of node kz+1; node kz gets 1-b
};
__device__ __forceinline__ AxW ax_own(int k, float b) { return AxW{k, b}; }
// staggered axial index from z - dz/2 (clamped at 0 as the reference does)
__device__ __forceinline__ AxW ax_half(int k, float b) {
  const bool down = b <= 0.5f && k > 0;
  return AxW{down ? k - 1 : k, down ? b + 0.5f : b - 0.5f};
}

// the four-node interpolation, its multiply-adds written out so that every
// field source rounds alike however its code is compiled; HZ: the order H_z
// is interpolated in
template <bool HZ = false>
__device__ __forceinline__ float stencil(float f00, float f01, float f10, float f11, RadW rw, AxW aw) {
  const float b = aw.b, ob = 1.f - aw.b;
  const float t0 = fmaf(f00, ob, f01 * b);
  if (HZ) return fmaf(rw.B, fmaf(f11, b, f10 * ob), t0 * rw.A);
  return fmaf(rw.A, t0, fmaf(f10, ob, f11 * b) * rw.B);
}

// node values are rounded to FP32 and multiplied by the push's scale s
// (escale for E, bscale for H) before the interpolation
template <bool HZ = false>
__device__ __forceinline__ float gather(const F32Args &p, const double *__restrict__ F, float s, RadW rw, AxW aw) {
  int ir = rw.ir, kz = aw.kz;
  if (ir > p.nr - 2 || kz > p.nz - 2) {
    atomicOr(p.err, kErrDomain);
    ir = min(ir, p.nr - 2);
    kz = min(kz, p.nz - 2);
  }
  const double *row0 = F + (size_t)ir * (size_t)p.nz + kz;
  const double *row1 = row0 + p.nz;
  float f00 = (float)row0[0] * s, f01 = (float)row0[1] * s, f10 = (float)row1[0] * s, f11 = (float)row1[1] * s;
  return stencil<HZ>(f00, f01, f10, f11, rw, aw);
}

// field sources of the push.  GlobalFields reads the six FP64 components
// from HBM / L2 per particle; BoxFields serves the particles of a cell-sorted
// block from an LDS copy (converted to FP32 once per node) of the nodes their
// cells can touch, and falls back to HBM for the rest.  Both evaluate the same
// FP32 expression on the same FP32-rounded node values; the result does not
// depend on the source but for H_z, which the tiles (BoxFields, TileGlobalFields)
// and an ensemble's bunches interpolate in another order than a single run's
// bunches (GlobalFields).  So a bunch particle alone and in an ensemble may differ
// by the rounding of its H_z; the orders are those that either has had all along.
// the two table entries of row i (the host builds p.rows with the same FP64
// expressions, so both give the same FP32 values)
__device__ __forceinline__ void row_entries(int i, float4 &t0, float4 &t1) {
  const double fi = i;
  t0 = make_float4(i ? (float)(1.0 / (2.0 * fi)) : 0.f, (float)(1.0 / (2.0 * (fi + 1))), (float)(1.0 / (2.0 * (fi + 2))),
                   (float)(1.0 / (2.0 * (fi + 3))));
  t1 = make_float4(i ? (float)(1.0 / fi) : 0.f, (float)(1.0 / (fi + 1)), (float)(1.0 / (fi + 0.5)), (float)(fi * (fi + 1)));
}

// (HZ: H_z in the order of the box's)
template <bool HZ>
struct GlobalFieldsT {
  __device__ __forceinline__ GlobalFieldsT() {}
  __device__ __forceinline__ GlobalFieldsT(const float *, int, int, int) {}
  // the two table entries of row i (clamped only for memory safety: a corrupt
  // cell word is caught by the gathers' domain check)
  __device__ __forceinline__ void row(const F32Args &p, int i, float4 &t0, float4 &t1) const {
    const int r = min(max(i, 0), p.nr - 1);
    t0 = p.rows[2 * r];
    t1 = p.rows[2 * r + 1];
  }
  __device__ __forceinline__ void get(const F32Args &p, int, int, RadW rl, RadW ro, AxW zo, AxW zh, float e[3],
                                      float h[3]) const {
    e[0] = gather(p, field(p, kER), p.escale, rl, zo);
    e[1] = gather(p, field(p, kEPhi), p.escale, ro, zo);
    e[2] = gather(p, field(p, kEZ), p.escale, ro, zh);
    h[0] = gather(p, field(p, kHHR), p.bscale, ro, zh);
    h[1] = gather(p, field(p, kHHPhi), p.bscale, rl, zh);
    h[2] = gather<HZ>(p, field(p, kHHZ), p.bscale, rl, zo);
  }
};
using GlobalFields = GlobalFieldsT<false>;
using TileGlobalFields = GlobalFieldsT<true>;

// rows bi..bi+kFR-1, columns bk..bk+width-1 of the six components, anchored
// two rows and two columns below the tile's anchor cell (ai, ak): a particle
// in cell (i, k) reads rows i-1..i+1 and columns k-1..k+1, so every cell with
// i in [ai-1, ai+1] and k in [ak-1, ak+width-4] is served from the box (a
// sorted tile lies along row ai; between sorts some of its particles have
// moved to the rows next to it, or to the column before its first).  width is
// kFK, or half of it for a tile that ends within the first half.  (With 64
// columns a 4096-particle tile overran the box below 66 particles per cell and
// its other particles gathered from HBM: the kernel on 4096-particle tiles at
// 40 per cell took 338 us for 2.1e7 particles, with 128 columns 238 us.)
// Components with the same stencil are stored together: {E_r, H_z} and
// {E_z, H_r} as pairs, E_phi and H_phi alone, so that a stencil is four
// addresses and eight LDS reads.
constexpr int kFR = 5, kFK = 128, kFComp = 6, kFPlane = kFR * kFK;
constexpr int kFBelow = 2;  // box rows and columns below the anchor cell
// the LDS array (floats): {E_r, H_z}, {E_z, H_r}, E_phi, H_phi, then two
// float4 row entries for each box row
constexpr int kFErHz = 0, kFEzHr = 2 * kFPlane, kFEphi = 4 * kFPlane, kFHphi = 5 * kFPlane, kFRows = 6 * kFPlane;
constexpr int kFBoxFloats = kFRows + 8 * kFR;

__device__ __forceinline__ float gather_box(const float *e, RadW rw, AxW aw) {
  return stencil(e[0], e[1], e[kFK], e[kFK + 1], rw, aw);
}

struct BoxFields {
  const float *box;  // LDS
  int ai, ak;        // anchor cell of the tile
  int width;         // columns filled
  __device__ __forceinline__ BoxFields(const float *b, int i, int k, int w) : box(b), ai(i), ak(k), width(w) {}
  // the box's row entries (an LDS read for every particle), replaced by the
  // entries evaluated in place for a row outside the box.  A global load here
  // would make the read a flat load, whose wait also waits for the next
  // particle's state loads already in flight.
  __device__ __forceinline__ void row(const F32Args &p, int i, float4 &t0, float4 &t1) const {
    const int li = i - ai + kFBelow;
    const int lc = min(max(li, 0), kFR - 1);
    const float4 *t = reinterpret_cast<const float4 *>(box + kFRows);
    t0 = t[2 * lc];
    t1 = t[2 * lc + 1];
    if ((unsigned)li >= (unsigned)kFR) row_entries(min(max(i, 0), p.nr - 1), t0, t1);
  }
  __device__ __forceinline__ void get(const F32Args &p, int i, int k, RadW rl, RadW ro, AxW zo, AxW zh, float e[3],
                                      float h[3]) const {
    const bool inbox = (unsigned)(i - ai + kFBelow - 1) < (unsigned)(kFR - 2) &&
                       (unsigned)(k - ak + kFBelow - 1) < (unsigned)(width - 2) && i <= p.nr - 2 && k <= p.nz - 2;
    if (inbox) {
      const int bi = ai - kFBelow, bk = ak - kFBelow;
      // the stencil's first entry for each (radial, axial) weight pair
      const int rlo = (rl.ir - bi) * kFK, roo = (ro.ir - bi) * kFK, zoo = zo.kz - bk, zho = zh.kz - bk;
      const float2 *erhz = reinterpret_cast<const float2 *>(box + kFErHz) + (rlo + zoo);
      const float2 *ezhr = reinterpret_cast<const float2 *>(box + kFEzHr) + (roo + zho);
      const float2 p00 = erhz[0], p01 = erhz[1], p10 = erhz[kFK], p11 = erhz[kFK + 1];
      const float e0 = stencil(p00.x, p01.x, p10.x, p11.x, rl, zo);
      const float h2 = stencil<true>(p00.y, p01.y, p10.y, p11.y, rl, zo);
      const float e1 = gather_box(box + kFEphi + (roo + zoo), ro, zo);
      const float2 q00 = ezhr[0], q01 = ezhr[1], q10 = ezhr[kFK], q11 = ezhr[kFK + 1];
      const float e2 = stencil(q00.x, q01.x, q10.x, q11.x, ro, zh);
      const float h0 = stencil(q00.y, q01.y, q10.y, q11.y, ro, zh);
      const float h1 = gather_box(box + kFHphi + (rlo + zho), rl, zh);
      e[0] = e0; e[1] = e1; e[2] = e2;
      h[0] = h0; h[1] = h1; h[2] = h2;
    } else {
      const float e0 = gather(p, field(p, kER), p.escale, rl, zo);
      const float e1 = gather(p, field(p, kEPhi), p.escale, ro, zo);
      const float e2 = gather(p, field(p, kEZ), p.escale, ro, zh);
      const float h0 = gather(p, field(p, kHHR), p.bscale, ro, zh);
      const float h1 = gather(p, field(p, kHHPhi), p.bscale, rl, zh);
      const float h2 = gather<true>(p, field(p, kHHZ), p.bscale, rl, zo);
      e[0] = e0; e[1] = e1; e[2] = e2;
      h[0] = h0; h[1] = h1; h[2] = h2;
    }
  }
};

// block prologue: fill the field box's first `width` columns (nodes outside
// the grid hold the nearest node's value; no particle that the box serves
// reads them).  One wavefront per 64 columns of a box row of one component,
// the kFComp * kFR rows dealt out evenly; a wave's loads are all in flight
// before the first is used (a branch or a use between them had made the
// prologue a chain of load latencies).
template <int WAVES>
__device__ __forceinline__ void field_box_fill(const F32Args &p, float *box, int ai, int ak, int width) {
  const int bi = ai - kFBelow, bk = ak - kFBelow;
  if (threadIdx.x < 2 * kFR) {
    const int r = min(max(bi + (int)(threadIdx.x >> 1), 0), p.nr - 1);
    reinterpret_cast<float4 *>(box + kFRows)[threadIdx.x] = p.rows[2 * r + (threadIdx.x & 1)];
  }
  constexpr int kLines = kFComp * kFR, kBatch = 8;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  for (int col = threadIdx.x & 63; col < width; col += 64) {
    const unsigned gk = min(max(bk + col, 0), p.nz - 1);
    for (int t0 = wave; t0 < kLines; t0 += WAVES * kBatch) {
      double v[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const int line = min(t0 + u * WAVES, kLines - 1), comp = line / kFR;
        const int gi = min(max(bi + line - comp * kFR, 0), p.nr - 1);
        // kHHR .. kHHZ are components 6 .. 8 of the grid
        v[u] = at(field(p, comp < 3 ? comp : comp + 3) + (size_t)gi * p.nz, gk * 8u);
      }
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const int line = t0 + u * WAVES, comp = line / kFR, row = line - comp * kFR;
        if (line >= kLines) break;
        // E_r, E_phi, E_z, H_r, H_phi, H_z
        const int plane = comp == 0 ? kFErHz : comp == 1 ? kFEphi : comp == 2 ? kFEzHr : comp == 3 ? kFEzHr + 1 : comp == 4 ? kFHphi : kFErHz + 1;
        const int step = comp == 1 || comp == 4 ? 1 : 2;
        box[plane + (row * kFK + col) * step] = (float)v[u] * (comp < 3 ? p.escale : p.bscale);
      }
    }
  }
}

__device__ __forceinline__ float dot3f(const float *a, const float *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

// relativistic Boris on u = gamma v, src/particles.cpp:1025-1150; e and h
// arrive multiplied by escale and bscale (the field sources apply them per node)
__device__ __forceinline__ void boris_u(const F32Args &p, const float e[3], const float h[3], float u[3]) {
  const float ee[3] = {e[0], e[1], e[2]};
  float b[3] = {h[0], h[1], h[2]};
  for (int j = 0; j < 3; j++) u[j] += ee[j];
  float g = frsq(1.f + dot3f(u, u) * p.inv_c2);
  for (int j = 0; j < 3; j++) b[j] *= g;
  float c2 = fdiv(2.f, 1.f + dot3f(b, b));
  float t0 = u[0], t1 = u[1], t2 = u[2];
  u[0] = t0 + c2 * ((t1 - t0 * b[2] + t2 * b[0]) * b[2] - (t2 + t0 * b[1] - t1 * b[0]) * b[1]);
  u[1] = t1 + c2 * (-(t0 + t1 * b[2] - t2 * b[1]) * b[2] + (t2 + t0 * b[1] - t1 * b[0]) * b[0]);
  u[2] = t2 + c2 * ((t0 + t1 * b[2] - t2 * b[1]) * b[1] - (t1 - t0 * b[2] + t2 * b[0]) * b[0]);
  for (int j = 0; j < 3; j++) u[j] += ee[j];
}

// Vay on u, src/particles.cpp:1152-1254 (with the reference's b scaling; e
// and h arrive multiplied by escale and bscale)
__device__ __forceinline__ void vay_u(const F32Args &p, const float e[3], const float h[3], float u[3]) {
  const float ee[3] = {e[0], e[1], e[2]};
  float b[3] = {h[0], h[1], h[2]};
  float t[3] = {u[0], u[1], u[2]};
  float g = frsq(1.f + dot3f(t, t) * p.inv_c2);
  float up[3];
  up[0] = t[0] + ee[0] + g * (t[1] * b[2] - t[2] * b[1]);
  up[1] = t[1] + ee[1] + g * (t[2] * b[0] - t[0] * b[2]);
  up[2] = t[2] + ee[2] + g * (t[0] * b[1] - t[1] * b[0]);
  float alpha = 1.f + dot3f(up, up) * p.inv_c2;  // gamma'^2
  float B2 = dot3f(b, b);
  float s = alpha - B2;
  const float ub = fmaf(up[2], b[2], fmaf(up[1], b[1], up[0] * b[0]));
  float us2 = ub * ub;
  float ig = frsq(0.5f * (s + fsqrt(s * s + 4.f * (B2 + us2))));  // 1/gamma^{n+1}
  for (int j = 0; j < 3; j++) b[j] *= ig;
  s = fdiv(1.f, 1.f + dot3f(b, b));
  alpha = dot3f(up, b);
  u[0] = s * (up[0] + alpha * b[0] + b[2] * up[1] - b[1] * up[2]);
  u[1] = s * (up[1] + alpha * b[1] + b[0] * up[2] - b[2] * up[0]);
  u[2] = s * (up[2] + alpha * b[2] + b[1] * up[0] - b[0] * up[1]);
}

// bring an offset back into (0, 1]: by ceil(o) - 1 cells (one cell at most
// after a half step; exact in FP32)
__device__ __forceinline__ void renorm(int &c, float &o) {
  const float m = ceilf(o) - 1.f;
  o -= m;
  c += (int)m;
}

// r of the Cartesian point (X, dy), X = i + xa, as an offset update that
// never forms X^2 + dy^2 - X^2: R - X = dy^2 / (R + X) for X > 0 (and
// R + |X| when the point lies behind the axis).  Returns sin(theta) = dy / R;
// ct = |X| / R is the reference's sqrt(1 - sin^2) (src/particles.cpp:1010).
__device__ __forceinline__ float rotate_back(int i, float &xa, float dy, float &ct) {
  const float X = (float)i + xa;
  const float s = fmaxf(X * X + dy * dy, 1e-30f);
  const float q = frsq(s);  // 1 / R
  const float R = s * q;
  xa += X > 0.f ? fdiv(dy * dy, R + X) : R - X;
  ct = fabsf(X) * q;
  return dy * q;
}

// J_phi of one particle at the half-step position,
// azimuthal_current_distribution (src/particles.cpp:688-784) in cell units
template <class S>
__device__ void deposit_jphi(const F32Args &p, S &sk, float w, int i, float a, int k, float b, float vphi) {
  double c0, c1;  // node (i,k) and (i+1,k) weights before the axial split
  if (i == 0) {
    double ad = a;  // axis cell in FP64; rho = a here
    c0 = 8.0 * (1.0 - ad);
    c1 = 1.0 + ad;
  } else {
    // 1 / (rho i) and 1 / (rho (i+1)) from one reciprocal
    const float fi = (float)i, rho = fi + a, fi1 = fi + 1.f;
    const float inv = __builtin_amdgcn_rcpf(rho * fi * fi1);
    c0 = (1.f - a) * (2.f * fi + a) * (fi1 * inv);
    c1 = a * (2.f * fi + 1.f + a) * (fi * inv);
  }
  float s = p.kp * w * vphi;
  const double s0 = (double)(s * (1.f - b)), s1 = (double)(s * b);
  sk.template add4<kCPhi>(i, k, s0 * c0, s0 * c1, s1 * c0, s1 * c1);
}

// Particles::charge_weighting of one particle (src/particles.cpp:101-226)
template <class S>
__device__ void deposit_rho(const F32Args &p, S &sk, float w, int i, float a, int k, float b) {
  double c0, c1;
  if (i == 0) {
    double rho = a;
    if (rho <= 0.5) {  // r <= dr/2 branch (:155-186)
      c0 = 16.0 * (0.5 - rho + rho * rho) / (2.0 * rho * rho + 0.5);
      c1 = 2.0 * rho * (rho + 1.0) / (2.0 * rho * rho + 0.5);
    } else {  // dr/2 < r <= dr (:188-218)
      c0 = 8.0 * (1.0 - rho);
      c1 = 1.0 + rho;
    }
  } else {
    const float fi = (float)i, rho = fi + a, fi1 = fi + 1.f;
    const float inv = __builtin_amdgcn_rcpf(rho * fi * fi1);
    c0 = (1.f - a) * (2.f * fi + a) * (fi1 * inv);
    c1 = a * (2.f * fi + 1.f + a) * (fi * inv);
  }
  float s = p.kp * w;
  const double s0 = (double)(s * (1.f - b)), s1 = (double)(s * b);
  sk.template add4<kCRho>(i, k, s0 * c0, s0 * c1, s1 * c0, s1 * c1);
}

// (log(1+x) - x) / x without cancellation
__device__ __forceinline__ float m_of(float x) {
  if (fabsf(x) < 0.1f)
    return x * (-0.5f + x * (1.f / 3.f + x * (-0.25f + x * (0.2f + x * (-1.f / 6.f + x * (1.f / 7.f - x * 0.125f))))));
  return fdiv(log1pf(x) - x, x);
}

// one straight piece of the path inside cell (i, k): simple_current_distribution
// (src/particles.cpp:333-474) rewritten in cell units.  (a, b): start offsets
// in the cell, (dr_, dz_): displacement in cells.  The closed forms
//   J_z[i]   ~ dz/i     [ (1-a)(2i+a)/rho - dr/2 + i(i+1)/rho M(x) ]
//   J_z[i+1] ~ dz/(i+1) [ a(2i+1+a)/rho  + dr/2 - i(i+1)/rho M(x) ]
//   J_r[k]   ~ [dr((1-b)/2 - dz/4) + i(i+1)/(2rho)(dr(1-b)/rho_e + dz N(x))] / (i+1/2)
//   J_r[k+1] ~ [dr(b/2 + dz/4)     + i(i+1)/(2rho)(dr b/rho_e     - dz N(x))] / (i+1/2)
// with rho = i + a, x = dr/rho, M = (ln(1+x)-x)/x, N = 1/(1+x) - ln(1+x)/x are
// algebraically identical to the reference's expressions (which evaluate them
// as differences of O(i) terms); they also reduce to strict_motion_weighting
// (:786-988) for purely axial or radial motion.
template <class S>
__device__ void segment(const F32Args &p, S &sk, float w, int i, int k, float a, float b, float drho, float dzeta,
                        const float4 &t) {
  float jz0, jz1, jr0, jr1;
  float f0 = 1.f, f1 = 1.f, fr = 1.f;  // factors of the J_z pair and of J_r
  if (i == 0) {
    double rs = a;  // axis cell in FP64
    jz0 = (float)(8.0 * (1.0 - 0.5 * drho - rs));
    jz1 = (float)(0.5 * drho + 1.0 + rs);
    jr0 = drho * (0.5f * (1.f - b) - 0.25f * dzeta) * 2.f;
    jr1 = drho * (0.5f * b + 0.25f * dzeta) * 2.f;
  } else {
    // t: second table entry of row i (1/i, 1/(i+1), 1/(i+1/2), i(i+1)); the
    // closed forms above, with 1/rho factored out of the J_z brackets
    const float fi = (float)i;
    const float rs = fi + a, re = rs + drho;
    // 1/rs, 1/re from one reciprocal
    const float q = __builtin_amdgcn_rcpf(rs * re);
    const float irs = re * q, ire = rs * q;
    const float ii = t.w;
    const float M = m_of(drho * irs);
    const float iiM = ii * M;
    const float N = -drho * ire - M;  // x / (1 + x) = drho / re
    const float hdr = 0.5f * drho;
    jz0 = fmaf(irs, fmaf(1.f - a, 2.f * fi + a, iiM), -hdr);
    jz1 = fmaf(irs, fmaf(a, 2.f * fi + 1.f + a, -iiM), hdr);
    const float cc = 0.5f * ii * irs, qdz = 0.25f * dzeta, dri = drho * ire, dN = dzeta * N, ub = 1.f - b;
    jr0 = fmaf(drho, fmaf(0.5f, ub, -qdz), cc * fmaf(dri, ub, dN));
    jr1 = fmaf(drho, fmaf(0.5f, b, qdz), cc * fmaf(dri, b, -dN));
    // the divisions by i, i+1 and i+1/2 go into the scale factors
    f0 = t.x;
    f1 = t.y;
    fr = t.z;
  }
  const float sz = p.kz * w * dzeta, sr = p.kr * w * fr;
  sk.template add2<kCZ>(i, k, (double)(jz0 * (sz * f0)), (double)(jz1 * (sz * f1)));
  sk.template add2<kCR>(i, k, (double)(sr * jr0), (double)(sr * jr1));
}

// the path parameter in [0, 1] at which a move of `d` cells reaches a face
// `f` cells away.  A move across a face can round to d = 0 in cell units: a
// particle 4e-9 cells above a face that ends 1e-9 cells below it has the new
// offset 1 - 1e-9, which is 1.0f, in the cell below, and the displacement
// (-1) + (1.0f - 4e-9) is 0.  The face is then taken at the start of the path
// (the deposited current is that of the part of the move that FP32 keeps).
__device__ __forceinline__ float cross_param(float f, float d) {
  return d != 0.f ? fminf(fmaxf(fdiv(f, d), 0.f), 1.f) : 0.f;
}

// current_distribution (src/particles.cpp:476-686): the straight path from
// the old to the new position, split at the cell faces it crosses (at most
// one radial and one axial face: |displacement| <= c dt <= dr/2), each piece
// deposited in its own cell
template <class S, class FS>
__device__ void deposit_j(const F32Args &p, S &sk, const FS &fs, float w, int io, float ao, int ko, float bo, int in_,
                          float an, int kn, float bn, float4 rt) {
  int di = in_ - io, dk = kn - ko;
  if (di < -1 || di > 1 || dk < -1 || dk > 1) {
    atomicOr(p.err, kErrDomain);
    return;
  }
  float drho = (float)di + (an - ao);
  float dzeta = (float)dk + (bn - bo);
  // pieces before the faces the path crosses, at the path parameters tr, tz
  // where it meets them (in old-cell units the radial face is at offset 1
  // (di=+1) or 0 (di=-1))
  int ci = io, ck = ko;
  float ca = ao, cb = bo;  // current start point, offsets in cell (ci, ck)
  if (di != 0 || dk != 0) {
    float tr = 2.f, tz = 2.f;
    if (di != 0) tr = cross_param((di > 0 ? 1.f : 0.f) - ao, drho);
    if (dk != 0) tz = cross_param((dk > 0 ? 1.f : 0.f) - bo, dzeta);
    float tprev = 0.f;
    for (int pass = 0; pass < 2; pass++) {
      bool rfirst = tr <= tz;
      float t = rfirst ? tr : tz;
      if (t > 1.f) break;
      float sd_r = (t - tprev) * drho, sd_z = (t - tprev) * dzeta;
      if (rfirst) {
        float fr = di > 0 ? 1.f : 0.f;
        segment(p, sk, w, ci, ck, ca, cb, fr - ca, sd_z, rt);
        ci += di;
        float4 rt0;
        fs.row(p, ci, rt0, rt);  // the field source's copy of the table (LDS in a tile)
        ca = di > 0 ? 0.f : 1.f;
        cb += sd_z;
        tr = 2.f;
      } else {
        float fz = dk > 0 ? 1.f : 0.f;
        segment(p, sk, w, ci, ck, ca, cb, sd_r, fz - cb, rt);
        ck += dk;
        cb = dk > 0 ? 0.f : 1.f;
        ca += sd_r;
        tz = 2.f;
      }
      tprev = t;
    }
  }
  // last piece to the new position
  segment(p, sk, w, ci, ck, ca, cb, (an + (float)(in_ - ci)) - ca, (bn + (float)(kn - ck)) - cb, rt);
}

// wall handling of move_half_reflect on the Cartesian half-step point
// (src/particles.cpp:1318-1353, src/bunch.cpp:126-153), in cell units: the
// walls sit at offset 1/2 of the first and last cells
__device__ __forceinline__ void walls(const F32Args &p, int &i, float &xa, int &k, float &b, float u[3],
                                      bool &alive) {
  // a point at least two cells from every wall cannot reach one (|offset
  // change| <= 1/4 per half step): nothing to test
  if (i >= 2 && i <= p.nr - 4 && k >= 2 && k <= p.nz - 4) return;
  const int il = p.nr - 2, kl = p.nz - 2;
  float off = (float)(i - il) + xa;
  if (i >= il - 1 && off > 0.5f) {
    if (p.is_bunch) {
      alive = false;
    } else {
      i = il;
      xa = 1.f - off;
      u[0] = -u[0];
    }
  }
  float offz = (float)(k - kl) + b;
  if (k >= kl - 1 && offz > 0.5f) {
    if (p.is_bunch) {
      alive = false;
    } else {
      k = kl;
      b = 1.f - offz;
      u[2] = -u[2];
    }
  }
  if (i <= 1) {
    float o0 = (float)i + xa;
    if (o0 < 0.5f) {
      i = 0;
      xa = 1.f - o0;
      u[0] = -u[0];
    }
  }
  if (k <= 1) {
    float o0 = (float)k + b;
    if (o0 < 0.5f) {
      k = 0;
      b = 1.f - o0;
      u[2] = -u[2];
    }
  }
}

// the state of one particle as loaded from HBM
struct PState {
  uint32_t c;
  float a, b, u0, u1, u2, w;
};

__device__ __forceinline__ PState load_state(const F32Args &p, unsigned off) {
  PState s;
  // streaming (non-temporal) loads and stores: each slot is touched once per
  // step, so the state should not displace the fields and tables from the caches
  s.c = __builtin_nontemporal_load(&at(p.cell, off));
  s.a = __builtin_nontemporal_load(&at(p.fa, off));
  s.b = __builtin_nontemporal_load(&at(p.fb, off));
  s.u0 = __builtin_nontemporal_load(&at(p.ur, off));
  s.u1 = __builtin_nontemporal_load(&at(p.uphi, off));
  s.u2 = __builtin_nontemporal_load(&at(p.uz, off));
  s.w = __builtin_nontemporal_load(&at(p.w, off));
  // all seven loads are issued together, ahead of the dead-particle branch
  // (instead of the six that the branch guards waiting for the cell word)
  asm volatile("" ::"v"(s.c), "v"(s.a), "v"(s.b), "v"(s.u0), "v"(s.u1), "v"(s.u2), "v"(s.w));
  return s;
}

// the state for the lane's next iteration: plain loads (they are waited for
// where the compiler needs them, or by wait_loads)
__device__ __forceinline__ PState load_state_next(const F32Args &p, unsigned off) {
  PState s;
  s.c = __builtin_nontemporal_load(&at(p.cell, off));
  s.a = __builtin_nontemporal_load(&at(p.fa, off));
  s.b = __builtin_nontemporal_load(&at(p.fb, off));
  s.u0 = __builtin_nontemporal_load(&at(p.ur, off));
  s.u1 = __builtin_nontemporal_load(&at(p.uphi, off));
  s.u2 = __builtin_nontemporal_load(&at(p.uz, off));
  s.w = __builtin_nontemporal_load(&at(p.w, off));
  return s;
}
// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima): every vector
// memory access of the wave has completed
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// the new state of one particle
struct POut {
  uint32_t c;
  float a, b, u0, u1, u2;
};

// the whole step of one particle (state ps) without its stores: false for a
// dead slot (nothing to store)
template <class S, class FS>
__device__ __forceinline__ bool step_state32(const F32Args &p, S &sk, const FS &fs, const PState &ps, POut &o) {
  const uint32_t c = ps.c;
  if (c & kDead) return false;
  int i = cell_i(c), k = cell_k(c);
  float a = ps.a, b = ps.b;
  float u[3] = {ps.u0, ps.u1, ps.u2};
  const float w = ps.w;
  sk.begin_cell(i, k);
  // gathers (E at the full step, H at the half-time copy)
  RadW rl, ro;
  float4 t0, t1;
  fs.row(p, i, t0, t1);
  rad_weights(i, a, t0, rl, ro);
  AxW zo = ax_own(k, b), zh = ax_half(k, b);
  float e[3], h[3];
  fs.get(p, i, k, rl, ro, zo, zh, e, h);
  if (p.pusher == 1)
    vay_u(p, e, h, u);
  else
    boris_u(p, e, h, u);
  float g = frsq(1.f + dot3f(u, u) * p.inv_c2);
  float dx = u[0] * g * p.hr, dy = u[1] * g * p.hr, dz = u[2] * g * p.hz;
  // first half step and rotation back to r-z (step_v, :1296-1316)
  int i1 = i, k1 = k;
  float xa = a + dx, b1 = b + dz;
  float ct;
  rotate_back(i1, xa, dy, ct);
  renorm(i1, xa);
  renorm(k1, b1);
  deposit_jphi(p, sk, w, i1, xa, k1, b1, u[1] * g);
  // second half step with the walls (move_half_reflect, :1355-1365)
  float xa2 = xa + dx, b2 = b1 + dz;
  bool alive = true;
  walls(p, i1, xa2, k1, b2, u, alive);
  const float st = rotate_back(i1, xa2, dy, ct);
  renorm(i1, xa2);
  renorm(k1, b2);
  if (alive) {
    deposit_j(p, sk, fs, w, i, a, k, b, i1, xa2, k1, b2, t1);
    // back_velocity_to_rz with the second half step's angle (:1005-1023)
    float u0 = ct * u[0] - st * u[1];
    float u1 = st * u[0] + ct * u[1];
    u[0] = u0;
    u[1] = u1;
    if (p.want_rho) deposit_rho(p, sk, w, i1, xa2, k1, b2);
  }
  o.c = pack(i1, k1) | (alive ? 0u : kDead);
  o.a = xa2;
  o.b = b2;
  o.u0 = u[0];
  o.u1 = u[1];
  o.u2 = u[2];
  return true;
}

__device__ __forceinline__ void store_state(const F32Args &p, const POut &o, unsigned off) {
  // a fresh copy of the offset: the stores then address from the scalar bases
  // too, instead of reusing 64-bit addresses formed for the loads
  unsigned so = off;
  asm("" : "+v"(so));
  __builtin_nontemporal_store(o.c, &at(p.cell, so));
  __builtin_nontemporal_store(o.a, &at(p.fa, so));
  __builtin_nontemporal_store(o.b, &at(p.fb, so));
  __builtin_nontemporal_store(o.u0, &at(p.ur, so));
  __builtin_nontemporal_store(o.u1, &at(p.uphi, so));
  __builtin_nontemporal_store(o.u2, &at(p.uz, so));
}

// the whole step of the particle in slot `slot` of the arrays of p (which
// start at most 2^30 slots before it)
template <class S, class FS>
__device__ __forceinline__ void step_particle32(const F32Args &p, S &sk, const FS &fs, unsigned slot) {
  POut o;
  if (step_state32(p, sk, fs, load_state(p, slot * 4u), o)) store_state(p, o, slot * 4u);
}

// the arguments with the particle arrays starting at slot `base` (uniform over
// the block): slots are then addressed by a 32-bit offset from a scalar base
__device__ __forceinline__ F32Args from_slot(const F32Args &p, long long base) {
  F32Args q = p;
  q.cell += base;
  q.fa += base;
  q.fb += base;
  q.ur += base;
  q.uphi += base;
  q.uz += base;
  q.w += base;
  return q;
}

// one tile of a cell-sorted (chunked) species from slot `base` (TileMap): its
// lanes read contiguous slots (coalesced) and each walks PPT consecutive
// logical particles, mostly of one cell.
template <int WAVES, class Map>
__device__ __forceinline__ void fused32_tile(const F32Args &p, const GlobalSink &gs, const Map &map, long long base,
                                             long long n_cap, double *box, float *fbox) {
  // one or two particles per lane: no register sums and no field box, whose
  // filling (15 to 30 loads a lane and a barrier) takes longer than the
  // particles' 24 loads each from L2
  using Sink = typename std::conditional<Map::kShort, TileSinkTall, TileSink>::type;
  using Fields = typename std::conditional<Map::kShort, TileGlobalFields, BoxFields>::type;
  const F32Args q = from_slot(p, base);
  const unsigned lim = (unsigned)min(n_cap - base, (long long)map.span());
  const unsigned off0 = map.first(threadIdx.x);
  // the lane's first particle is on its way while the boxes are set up
  PState nx{kDead, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (off0 < lim) nx = load_state_next(q, off0 * 4u);
  Sink sk;
  int ai = 0, ak = 0, width = 0;
  if constexpr (Map::kShort) {
    tall_init(box, cell_i(nx.c), cell_k(nx.c), !(nx.c & kDead), Map::kParticles, p.n, sk, gs);
  } else {
    static_assert(kFK == Sink::kK, "the two boxes share their width");
    // anchor samples: slot base + j is the logical particle 16 j of the tile
    bool live[3];
    int ri[3], kk[3];
#pragma unroll
    for (int j = 0; j < 3; j++) {
      const uint32_t c = base + j < n_cap ? p.cell[base + j] : kDead;
      live[j] = !(c & kDead);
      ri[j] = cell_i(c);
      kk[j] = cell_k(c);
    }
    tile_anchor(live, ri, kk, ai, ak);
    // the boxes' width: half of it when the tile's last particle (the last
    // slot its threads reach) lies within the first half of the anchor's row,
    // with one column to spare
    const uint32_t cl = base + map.last() < n_cap ? p.cell[base + map.last()] : kDead;
    const bool narrow = !(cl & kDead) && cell_i(cl) == ai && cell_k(cl) - ak <= kFK / 2 - 5;
    width = narrow ? kFK / 2 : kFK;
    box_init(box, ai, ak, width, sk, gs);
    field_box_fill<WAVES>(p, fbox, ai, ak, width);
    __syncthreads();
  }
  const Fields fs(fbox, ai, ak, width);
  // software pipeline: the state of the lane's next particle is loaded before
  // the current one is pushed; all its loads are waited for before the
  // current particle's stores, so the wait never includes stores in flight
  for (int j = 0; j < map.ppt(); j++) {
    const PState cur = nx;
    unsigned n = off0 + (unsigned)j * 64u, n1 = n + 64u;
    asm("" : "+v"(n), "+v"(n1));  // keeps the slots 32-bit offsets from the scalar bases (no 64-bit pointer per array)
    if (j + 1 < map.ppt() && n1 < lim) nx = load_state_next(q, n1 * 4u);
    POut o;
    const bool st = n < lim && step_state32(q, sk, fs, cur, o);
    wait_loads();
    if (st) store_state(q, o, n * 4u);
  }
  sk.flush();
  __syncthreads();
  box_flush(box, sk);
}

template <int PPT, int WAVES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) k_fused32_tiled(F32Args p, GlobalSink gs, long long n_cap) {
  __shared__ double box[PPT <= 2 ? TileSinkTall::kSize : TileSink::kSize];
  __shared__ __align__(16) float fbox[kFBoxFloats];
  // launched for the chunked layout only, i.e. plasma species: no bunch walls
  // and no charge density (constants here drop their code and registers)
  F32Args q = p;
  q.is_bunch = 0;
  q.want_rho = 0;
  // the sink's grid size and error word are the arguments' (one copy each in
  // scalar registers)
  GlobalSink g = gs;
  g.nr = q.nr;
  g.nz = q.nz;
  g.err = q.err;
  using Map = TileMap<PPT, WAVES>;
  fused32_tile<WAVES>(q, g, Map(), Map::base(blockIdx.x), n_cap, box, fbox);
}

// one block of a bunch (plain layout): WAVES x 64 x PPT slots from `base`; the
// box takes the shape that suits the cells of the block's living particles
// (bunch_init)
template <int WAVES, int PPT, class Fields = GlobalFields>
__device__ __forceinline__ void fused32_bunch_tile(const F32Args &p, const GlobalSink &gs, long long base,
                                                   long long n_cap, double *box) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long cbase = base + (long long)wave * (64 * PPT) + lane;
  int i0 = 0x7fffffff, k0 = 0x7fffffff, i1 = -1, k1 = -1;
  for (int j = 0; j < PPT; j++) {
    long long n = cbase + (long long)j * 64;
    if (n < n_cap) {
      uint32_t c = p.cell[n];
      if (!(c & kDead)) {
        const int i = cell_i(c), k = cell_k(c);
        i0 = min(i0, i);
        k0 = min(k0, k);
        i1 = max(i1, i);
        k1 = max(k1, k);
      }
    }
  }
  // (neighbouring slots of a bunch are not in one cell: register sums help
  // only where a lane walks several)
  using Sink = typename std::conditional<PPT == 1, BunchSinkOne, BunchSink>::type;
  Sink sk;
  if (!bunch_init<WAVES>(box, i0, k0, i1, k1, sk, gs)) return;
  const F32Args q = from_slot(p, base);
  const unsigned lim = (unsigned)min(n_cap - base, (long long)WAVES * 64 * PPT);
  const unsigned off0 = (unsigned)(wave * 64 * PPT + lane);
  for (int j = 0; j < PPT; j++) {
    const unsigned n = off0 + (unsigned)j * 64u;
    if (n < lim) step_particle32(q, sk, Fields(), n);
  }
  sk.flush();
  __syncthreads();
  box_flush(box, sk);
}

// bunches: PPT particles per lane (wave w of a block takes the 64 * PPT slots
// from w * 64 * PPT); a small bunch takes few per lane so that its blocks
// still spread over the GPU
template <int PPT>
__global__ void __launch_bounds__(256) k_fused32_bunch(F32Args p, GlobalSink gs, long long n_cap) {
  __shared__ double box[BunchSink::kSize];
  fused32_bunch_tile<kWavesPerBlock, PPT>(p, gs, (long long)blockIdx.x * (kWavesPerBlock * 64 * PPT), n_cap, box);
}

// A pointer read from device memory is generic (flat) to the compiler: its
// loads, stores and atomics become flat instructions on 64-bit per-lane
// addresses, which also hold up the kernel's LDS waits.  The ensemble's
// argument tables are therefore read through mirrors of F32Args and
// GlobalSink whose pointers are in the global address space (same layout);
// converted to the generic structs, every access derived from them compiles
// to global instructions on scalar bases, as for kernel arguments.
template <class T>
using gptr = __attribute__((address_space(1))) T *;
struct F32ArgsG {
  int nr, nz;
  float hr, hz, inv_c2, c1, bscale, escale, kz, kr, kp;
  int pusher, is_bunch, want_rho, n;
  gptr<const double> grid;
  gptr<const float4> rows;
  gptr<int> err;
  gptr<uint32_t> cell;
  gptr<float> fa, fb, ur, uphi, uz;
  gptr<const float> w;
};
static_assert(sizeof(F32ArgsG) == sizeof(F32Args) && offsetof(F32ArgsG, grid) == offsetof(F32Args, grid) &&
                  offsetof(F32ArgsG, w) == offsetof(F32Args, w) && offsetof(F32ArgsG, n) == offsetof(F32Args, n),
              "F32ArgsG mirrors F32Args");
struct GlobalSinkG {
  int nr, nz;
  gptr<double> j, rho;
  gptr<int> err;
};
static_assert(sizeof(GlobalSinkG) == sizeof(GlobalSink) && offsetof(GlobalSinkG, err) == offsetof(GlobalSink, err),
              "GlobalSinkG mirrors GlobalSink");

__device__ __forceinline__ F32Args from_global(const F32ArgsG &g) {
  F32Args a;
  a.nr = g.nr;
  a.nz = g.nz;
  a.hr = g.hr;
  a.hz = g.hz;
  a.inv_c2 = g.inv_c2;
  a.c1 = g.c1;
  a.bscale = g.bscale;
  a.escale = g.escale;
  a.kz = g.kz;
  a.kr = g.kr;
  a.kp = g.kp;
  a.pusher = g.pusher;
  a.is_bunch = g.is_bunch;
  a.want_rho = g.want_rho;
  a.n = g.n;
  a.grid = (const double *)g.grid;
  a.rows = (const float4 *)g.rows;
  a.err = (int *)g.err;
  a.cell = (uint32_t *)g.cell;
  a.fa = (float *)g.fa;
  a.fb = (float *)g.fb;
  a.ur = (float *)g.ur;
  a.uphi = (float *)g.uphi;
  a.uz = (float *)g.uz;
  a.w = (const float *)g.w;
  return a;
}
__device__ __forceinline__ GlobalSink from_global(const GlobalSinkG &g) {
  GlobalSink s;
  s.nr = g.nr;
  s.nz = g.nz;
  s.j = (double *)g.j;
  s.rho = (double *)g.rho;
  s.err = (int *)g.err;
  return s;
}

// The species of one simulation in one launch: where none of them fills the
// GPU a launch is bound by the latency of its blocks (a 1e3-particle bunch
// takes 11.0 us, a 1.6e5-particle plasma 11.3, both in one launch 12.1).
// first[s]: the first block of species s; the bunches come first, their
// blocks (one particle per lane, global gathers) take the longest.
struct F32Group {
  F32ArgsG a[kMaxGroup];
  GlobalSinkG sink;
  int first[kMaxGroup];
  long long n_cap[kMaxGroup];
};

template <int PPT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) k_fused32_group(F32Group g) {
  constexpr int kBunch = BunchSink::kSize, kTile = TileSink::kSize + (kFBoxFloats + 1) / 2;
  __shared__ __align__(16) double lds[kBunch > kTile ? kBunch : kTile];
  static_assert(TileSink::kSize % 2 == 0, "the field box behind the current box is 16-byte aligned");
  static_assert(TileSinkTall::kSize <= kTile, "a small tile's box takes the place of both");
  int s = 0;
#pragma unroll
  for (int t = 1; t < kMaxGroup; t++) s += (int)blockIdx.x >= g.first[t] ? 1 : 0;
  F32Args p = from_global(g.a[s]);
  GlobalSink gs = from_global(g.sink);
  gs.nr = p.nr;
  gs.nz = p.nz;
  gs.err = p.err;
  const long long block = (int)blockIdx.x - g.first[s];
  if (p.is_bunch) {
    fused32_bunch_tile<kWavesPerBlock, 1>(p, gs, block * (kWavesPerBlock * 64), g.n_cap[s], lds);
  } else {
    p.want_rho = 0;
    using Map = TileMap<PPT, kWavesPerBlock>;
    fused32_tile<kWavesPerBlock>(p, gs, Map(), Map::base(block), g.n_cap[s], lds,
                                 reinterpret_cast<float *>(lds + TileSink::kSize));
  }
}

// ensembles: the plasma tiles and bunch blocks of every instance in one
// launch, one block per item of the work list (a persistent grid striding
// over the list kept the loop's state in scalar registers, which spilled).
// The tiles of a list may differ in size; its bunch blocks, the longest for
// their particles (gathers from HBM), come first and hold one particle per
// lane.  16 instances, 1.27e8 particles at 12 to 40 per cell, MI355X: 1646 us;
// with the bunches on the tiles' walk (4096 particles each, mostly past the
// boxes) and the sparse species in a launch of their own 1739 + 91 us.
struct EnsItem {
  int arg;   // index into the per-(instance, species) argument tables
  int lg;    // plasma tile of 2^lg particles per lane; -1: bunch block, one per lane
  long long base, n_cap;
};

// 5 waves per SIMD (96 VGPRs) once the table pointers are global; with flat
// pointers it needed 121 VGPRs and ran at 4
template <int WAVES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5)))
k_ens_fused32(const F32Args *__restrict__ args, const GlobalSink *__restrict__ sinks,
              const EnsItem *__restrict__ items, int n_items) {
  constexpr int kBunch = BunchSink::kSize, kTile = TileSink::kSize + (kFBoxFloats + 1) / 2;
  __shared__ __align__(16) double lds[kBunch > kTile ? kBunch : kTile];
  const int it = blockIdx.x;
  if (it >= n_items) return;
  const EnsItem item = items[it];
  const F32ArgsG *ag = reinterpret_cast<const F32ArgsG *>(args) + item.arg;
  const GlobalSinkG *sg = reinterpret_cast<const GlobalSinkG *>(sinks) + item.arg;
  F32Args a = from_global(*ag);
  GlobalSink g = from_global(*sg);
  g.nr = a.nr;  // one copy of the grid size and error word (scalar registers)
  g.nz = a.nz;
  g.err = a.err;
  if (item.lg < 0) {
    a.is_bunch = a.want_rho = 1;
    fused32_bunch_tile<WAVES, 1, TileGlobalFields>(a, g, item.base, item.n_cap, lds);
  } else {
    a.is_bunch = a.want_rho = 0;
    fused32_tile<WAVES>(a, g, TileMapRt<WAVES>{item.lg}, item.base, item.n_cap, lds,
                        reinterpret_cast<float *>(lds + TileSink::kSize));
  }
}

__global__ void k_charge32(F32Args p, GlobalSink gs, long long n_cap) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= n_cap) return;
  uint32_t c = p.cell[n];
  if (c & kDead) return;
  GlobalSink sk = gs;
  deposit_rho(p, sk, p.w[n], cell_i(c), p.fa[n], cell_k(c), p.fb[n]);
}

// plasma species: tiles of the chunked layout (k_charge32's four global
// atomics a particle, 20 of them on each node, took 401 us for 1.05e7
// particles)
template <int PPT>
__global__ void __launch_bounds__(256) k_charge32_tiled(F32Args p, GlobalSink gs, long long n_cap) {
  __shared__ double box[NodeSink::kSize];
  using Map = TileMap<PPT, kWavesPerBlock>;
  const long long base = Map::base(blockIdx.x);
  int ai, ak;
  {
    bool live[3];
    int ri[3], kk[3];
#pragma unroll
    for (int j = 0; j < 3; j++) {
      const uint32_t c = p.cell[base + j];
      live[j] = !(c & kDead);
      ri[j] = cell_i(c);
      kk[j] = cell_k(c);
    }
    tile_anchor(live, ri, kk, ai, ak);
  }
  NodeSink sk;
  sk.init(gs, gs.rho, box, ai, ak);
  __syncthreads();
  const long long first = base + Map::first(threadIdx.x);
#pragma unroll
  for (int j = 0; j < PPT; j++) {
    const long long n = first + j * 64;
    const uint32_t c = p.cell[n];
    const float w = p.w[n], a = p.fa[n], b = p.fb[n];
    if (c & kDead) continue;
    sk.begin_cell(cell_i(c), cell_k(c));
    deposit_rho(p, sk, w, cell_i(c), a, cell_k(c), b);
  }
  sk.flush();
  __syncthreads();
  sk.to_grid();
}

// absolute FP64 state in logical order -> cell form in the species' layout
// (cell index by CELL_NUMBER clamped at 0; chunk padding slots marked)
__global__ void k_pack(GridDesc g, const double *r, const double *z, const double *vr, const double *vphi,
                       const double *vz, const double *w, const uint8_t *alive, int n, long long n_cap, int chunked,
                       uint32_t *cell, float *fa, float *fb, float *ur, float *uphi, float *uz, float *fw) {
  const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_cap) return;
  const long long j = chunked ? logical_of(p) : p;
  if (j >= n) {
    cell[p] = kPadCell;
    fa[p] = fb[p] = 0.5f;
    ur[p] = uphi[p] = uz[p] = fw[p] = 0.f;
    return;
  }
  double xr = r[j] / g.dr, xz = z[j] / g.dz;
  int i = (int)ceil(xr) - 1, k = (int)ceil(xz) - 1;
  if (i < 0) i = 0;
  if (k < 0) k = 0;
  if (i > g.nr - 2) i = g.nr - 2;
  if (k > g.nz - 2) k = g.nz - 2;
  float oa = (float)(xr - i), ob = (float)(xz - k);
  double v2 = vr[j] * vr[j] + vphi[j] * vphi[j] + vz[j] * vz[j];
  double gam = 1.0 / sqrt(1.0 - v2 / (kLightSpeed * kLightSpeed));
  cell[p] = pack(i, k) | (alive[j] == 1 ? 0u : kDead);
  fa[p] = oa;
  fb[p] = ob;
  ur[p] = (float)(gam * vr[j]);
  uphi[p] = (float)(gam * vphi[j]);
  uz[p] = (float)(gam * vz[j]);
  fw[p] = (float)w[j];
}

__global__ void k_unpack(GridDesc g, double *r, double *z, double *vr, double *vphi, double *vz, double *w,
                         uint8_t *alive, int n, int chunked, const uint32_t *cell, const float *fa, const float *fb,
                         const float *ur, const float *uphi, const float *uz, const float *fw) {
  const long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const long long p = chunked ? phys_of(j) : j;
  uint32_t c = cell[p];
  r[j] = ((double)cell_i(c) + (double)fa[p]) * g.dr;
  z[j] = ((double)cell_k(c) + (double)fb[p]) * g.dz;
  double u0 = ur[p], u1 = uphi[p], u2 = uz[p];
  double ig = 1.0 / sqrt(1.0 + (u0 * u0 + u1 * u1 + u2 * u2) / (kLightSpeed * kLightSpeed));
  vr[j] = u0 * ig;
  vphi[j] = u1 * ig;
  vz[j] = u2 * ig;
  w[j] = fw[p];
  alive[j] = (c & kDead) ? 0 : 1;
}

// Bunch::bunch_inject (src/bunch.cpp:104-121) on the cell form: z from the
// draw, v_z set to the bunch speed, the radial state kept
__device__ __forceinline__ void inject_one32(const GridDesc &g, uint32_t *cell, float *fb, float *ur, float *uphi,
                                             float *uz, const double *u, unsigned j, double dl, double velocity) {
  double zabs = dl * u[j] + g.dz / 2.0;
  double xz = zabs / g.dz;
  int k = (int)ceil(xz) - 1;
  if (k < 0) k = 0;
  uint32_t c = cell[j];
  double u0 = ur[j], u1 = uphi[j], u2 = uz[j];
  double ig = 1.0 / sqrt(1.0 + (u0 * u0 + u1 * u1 + u2 * u2) / (kLightSpeed * kLightSpeed));
  double v0 = u0 * ig, v1 = u1 * ig, v2 = velocity;
  double gam = 1.0 / sqrt(1.0 - (v0 * v0 + v1 * v1 + v2 * v2) / (kLightSpeed * kLightSpeed));
  cell[j] = pack(cell_i(c), k);
  fb[j] = (float)(xz - k);
  ur[j] = (float)(gam * v0);
  uphi[j] = (float)(gam * v1);
  uz[j] = (float)(gam * v2);
}
__global__ void k_inject32(GridDesc g, uint32_t *cell, float *fb, float *ur, float *uphi, float *uz,
                           const double *u, int n, unsigned start, unsigned count, double dl, double velocity) {
  unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  unsigned j = t + start;
  if (j >= (unsigned)n) return;
  inject_one32(g, cell, fb, ur, uphi, uz, u, j, dl, velocity);
}

// ensembles: the injections of every (instance, bunch) pair for the
// ensemble's current step, read from the step counter on the device (so the
// launch can sit in the step's graph); item y of the grid, particle x
__global__ void k_ens_inject(const EnsInjectItem *__restrict__ items, const long long *__restrict__ step) {
  const EnsInjectItem &it = items[blockIdx.y];
  const long long s = *step;
  if (s >= it.table_len) return;
  const int start = it.start[s];
  if (start < 0) return;
  for (unsigned t = blockIdx.x * blockDim.x + threadIdx.x; t < (unsigned)it.count; t += gridDim.x * blockDim.x) {
    const unsigned j = t + (unsigned)start;
    if (j >= (unsigned)it.n) break;
    inject_one32(it.g, it.cell, it.fb, it.ur, it.uphi, it.uz, it.u, j, it.dl, it.velocity);
  }
}
__global__ void k_ens_count(long long *step) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *step += 1;
}

F32Args args32(Ctx &c, Species &sp) {
  F32Args p;
  const GridDesc &g = c.g;
  p.nr = g.nr;
  p.nz = g.nz;
  p.hr = (float)(g.dt / (2.0 * g.dr));
  p.hz = (float)(g.dt / (2.0 * g.dz));
  p.inv_c2 = (float)(1.0 / (kLightSpeed * kLightSpeed));
  double c1 = sp.charge * g.dt / (2.0 * sp.mass);
  p.c1 = (float)c1;
  if (c.pusher == 1) {
    p.escale = (float)(2.0 * c1);
    p.bscale = (float)(kMagnConst * c1 * 2.0 * c1 * c1);
  } else {
    p.escale = (float)c1;
    p.bscale = (float)(kMagnConst * c1);
  }
  p.kz = (float)(sp.charge / (4.0 * kPi * g.dr * g.dr * g.dt));
  p.kr = (float)(sp.charge / (2.0 * kPi * g.dr * g.dz * g.dt));
  p.kp = (float)(sp.charge / (4.0 * kPi * g.dz * g.dr * g.dr));
  p.pusher = c.pusher;
  p.is_bunch = sp.kind == 1;
  p.want_rho = sp.kind == 1;
  p.n = sp.n;
  p.grid = c.grid;
  p.rows = c.rows;
  p.err = c.err;
  p.cell = (uint32_t *)sp.f32.cell;
  p.fa = sp.f32.fr;
  p.fb = sp.f32.fz;
  p.ur = sp.f32.vr;
  p.uphi = sp.f32.vphi;
  p.uz = sp.f32.vz;
  p.w = sp.f32.w;
  return p;
}

GlobalSink sink32(Ctx &c) {
  GlobalSink gs;
  gs.nr = c.g.nr;
  gs.nz = c.g.nz;
  gs.j = c.a[kJR];
  gs.rho = c.a[kRhoBunch];
  gs.err = c.err;
  return gs;
}

bool ensure_f32(Species &sp) {
  if (sp.f32.cell) return true;
  size_t n = sp.n_cap > 0 ? (size_t)sp.n_cap : 1;
  bool ok = hipMalloc((void **)&sp.f32.cell, n * sizeof(int32_t)) == hipSuccess;
  ok = ok && hipMalloc((void **)&sp.f32.fr, n * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&sp.f32.fz, n * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&sp.f32.vr, n * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&sp.f32.vphi, n * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&sp.f32.vz, n * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&sp.f32.w, n * sizeof(float)) == hipSuccess;
  return ok;
}

unsigned blocks_for(long long n) { return (unsigned)((n + 255) / 256); }

constexpr int kChunkTile = kNumTiles - 1;  // 4 x 4: one chunk per tile (the next shapes: 2 x 4 and 1 x 4)
static_assert(kTileShapes[kChunkTile][0] * kTileShapes[kChunkTile][1] == kPPT, "one-chunk tile shape");

}  // namespace

template <int PPT, int WAVES>
void launch_tile_t(hipStream_t st, const F32Args &p, const GlobalSink &gs, long long n_cap) {
  constexpr long long kTile = TileMap<PPT, WAVES>::kParticles;
  unsigned blocks = (unsigned)((n_cap + kTile - 1) / kTile);
  hipLaunchKernelGGL((k_fused32_tiled<PPT, WAVES>), dim3(blocks), dim3(WAVES * 64), 0, st, p, gs, n_cap);
}

void launch_tile(int tile, hipStream_t st, const F32Args &p, const GlobalSink &gs, long long n_cap) {
  switch (tile) {
    case 0: launch_tile_t<16, 4>(st, p, gs, n_cap); break;
    case 1: launch_tile_t<16, 2>(st, p, gs, n_cap); break;
    case 2: launch_tile_t<16, 1>(st, p, gs, n_cap); break;
    case 3: launch_tile_t<8, 4>(st, p, gs, n_cap); break;
    case 4: launch_tile_t<8, 2>(st, p, gs, n_cap); break;
    case 5: launch_tile_t<4, 4>(st, p, gs, n_cap); break;
    case 6: launch_tile_t<2, 4>(st, p, gs, n_cap); break;
    default: launch_tile_t<1, 4>(st, p, gs, n_cap); break;
  }
}

// the shape for a species of a context whose shape was neither set nor
// autotuned: of the shapes with boxes the largest that covers at most kFK - 8
// cells of a sorted species (its boxes then serve all of its particles) and has
// enough blocks for its long walk (sixteen on each of 256 CUs, or six of 4x4);
// smaller species run on the shapes without boxes, two particles per lane where
// that leaves three blocks on each CU, else one.  Kernel times in us right after a
// sort, shapes 16x4, 8x4, 4x4, 2x4, 1x4:
//   1.6e5 particles, 10 per cell:   56     35     23     12.2   10.9
//   1.0e6 twice, 13 per cell (Vay):  -      -     49     42      -
//   2.6e6 particles, 20 per cell:   79     58     50     59      -
//   2.1e7 particles, 40 per cell:  238    273    303      -      -
//   2.1e8 particles, 100 per cell: 2126  2432   2866      -      -
// and of the whole step 5 to 45 steps after it (500 eV: most lanes meet another
// cell with every particle):
//   1.6e5 particles, 10 per cell:  107      -     35     24     21
//   6.6e5 particles, 40 per cell:  108      -     45     37     43
//   9.8e5 particles, 15 per cell:  133      -     61     48     51
//   2.6e6 particles, 20 per cell:  248    108    101     93     97
//   7.9e6 particles, 30 per cell:  325    226    220    218      -
//   2.1e7 particles, 40 per cell:  529    499    516    556    580
// A species that has not been sorted for kDrift steps runs on the shapes without
// boxes whatever its size: its particles have drifted off the rows and columns
// that the larger tiles' boxes hold (1 eV, steps of half a cell at c, 10-step passes:
// 4e6 particles at 20 per cell 2.0 ms in order on 4x4 and 2.2 on 2x4, 5.6 and 2.5
// after 2000 steps; two species of 1.35e7 at 45 per cell 4.8 on 8x4 and 5.8, 14.2
// and 6.5; the lines cross after about 400 and 800 steps).  A hotter plasma drifts
// off sooner: the count of steps is late for it, and no worse than one shape for
// all.  Loaded in no order the shapes do not matter (2.1e7: 7514 and 7506 us): the
// deposits wait for the grid.
constexpr long long kDrift = 500;
int auto_tile(const Ctx &c, const Species &sp) {
  const double cells = (double)(c.g.nr - 1) * (c.g.nz - 1);
  const struct {
    int tile, particles, blocks;
  } shapes[] = {{0, 4096, 4096}, {3, 2048, 4096}, {5, 1024, 1536}};
  for (const auto &s : shapes)
    if (sp.steps_unsorted <= kDrift && sp.n >= (long long)s.particles * s.blocks && s.particles * cells <= (kFK - 8) * (double)sp.n) return s.tile;
  return sp.n >= 512 * 768 ? 6 : 7;
}

void launch_fused_f32(Ctx &c, Species &sp) {
  if (sp.n_cap <= 0 || !sp.f32.cell) return;
  if (sp.chunked) {
    launch_tile(c.tile_auto ? auto_tile(c, sp) : c.tile, c.stream, args32(c, sp), sink32(c), sp.n_cap);
  } else {
    // the most particles per lane that still give 1024 blocks
    const long long n = sp.n_cap, per = (long long)kWavesPerBlock * 64;
    const F32Args a = args32(c, sp);
    const GlobalSink g = sink32(c);
    if (n >= 1024 * per * kPPT)
      hipLaunchKernelGGL(k_fused32_bunch<kPPT>, dim3((unsigned)((n + per * kPPT - 1) / (per * kPPT))), dim3(256), 0,
                         c.stream, a, g, n);
    else if (n >= 1024 * per * 4)
      hipLaunchKernelGGL(k_fused32_bunch<4>, dim3((unsigned)((n + per * 4 - 1) / (per * 4))), dim3(256), 0, c.stream,
                         a, g, n);
    else
      hipLaunchKernelGGL(k_fused32_bunch<1>, dim3((unsigned)((n + per - 1) / per)), dim3(256), 0, c.stream, a, g, n);
  }
}

template <int PPT>
void launch_group_t(hipStream_t st, const F32Group &g, int blocks) {
  hipLaunchKernelGGL(k_fused32_group<PPT>, dim3(blocks), dim3(256), 0, st, g);
}

bool launch_group_f32(Ctx &c) {
  F32Group g;
  int n = 0, tile = -1;
  long long blocks = 0;
  // bunches, then plasma species
  for (int kind = 1; kind >= 0; kind--)
    for (int j : c.order) {
      Species &sp = c.species[j];
      if (sp.n_cap <= 0 || !sp.f32.cell || (sp.kind == 1) != (kind == 1)) continue;
      if (n == kMaxGroup) return false;
      long long per = kWavesPerBlock * 64;
      if (sp.chunked) {
        // one shape, of at most a chunk, for all plasma species
        const int t = c.tile_auto ? auto_tile(c, sp) : c.tile;
        if (t < kChunkTile || (tile >= 0 && t != tile)) return false;
        tile = t;
        per *= t == kChunkTile ? 4 : t == kChunkTile + 1 ? 2 : 1;
      } else if (sp.n_cap >= 1024 * per * 4) {
        return false;  // a bunch that walks several particles per lane
      }
      const F32Args a = args32(c, sp);
      memcpy(&g.a[n], &a, sizeof(a));
      g.first[n] = (int)blocks;
      g.n_cap[n] = sp.n_cap;
      blocks += (sp.n_cap + per - 1) / per;
      n++;
    }
  if (n < 2 || tile < 0 || blocks > 0x7fffffff) return false;
  for (int t = n; t < kMaxGroup; t++) g.first[t] = 0x7fffffff;
  const GlobalSink gs = sink32(c);
  memcpy(&g.sink, &gs, sizeof(gs));
  if (tile == kChunkTile)
    launch_group_t<4>(c.stream, g, (int)blocks);
  else if (tile == kChunkTile + 1)
    launch_group_t<2>(c.stream, g, (int)blocks);
  else
    launch_group_t<1>(c.stream, g, (int)blocks);
  return true;
}

void launch_charge_weighting_f32(Ctx &c, Species &sp, double *rho) {
  if (sp.n_cap <= 0 || !sp.f32.cell) return;
  GlobalSink gs = sink32(c);
  if (rho) gs.rho = rho;
  if (sp.chunked && sp.n_cap >= kOneChunkBlocks * kChunk)
    hipLaunchKernelGGL(k_charge32_tiled<4>, dim3((unsigned)(sp.n_cap / kChunk)), dim3(256), 0, c.stream, args32(c, sp), gs,
                       sp.n_cap);
  else if (sp.chunked)
    hipLaunchKernelGGL(k_charge32_tiled<1>, dim3((unsigned)(sp.n_cap / 256)), dim3(256), 0, c.stream, args32(c, sp), gs,
                       sp.n_cap);
  else
    hipLaunchKernelGGL(k_charge32, dim3(blocks_for(sp.n_cap)), dim3(256), 0, c.stream, args32(c, sp), gs, sp.n_cap);
}

void launch_bunch_inject_f32(Ctx &c, Species &sp, unsigned start, unsigned count, double dl) {
  if (count == 0 || !sp.f32.cell) return;
  hipLaunchKernelGGL(k_inject32, dim3((count + 255) / 256), dim3(256), 0, c.stream, c.g,
                     (uint32_t *)sp.f32.cell, sp.f32.fz, sp.f32.vr, sp.f32.vphi, sp.f32.vz, sp.inject_u, sp.n,
                     start, count, dl, sp.velocity);
}

bool launch_f32_from_f64(Ctx &c, Species &sp) {
  if (sp.n_cap <= 0) return true;
  if (!ensure_f32(sp)) return false;
  hipLaunchKernelGGL(k_pack, dim3(blocks_for(sp.n_cap)), dim3(256), 0, c.stream, c.g, sp.f64.r, sp.f64.z, sp.f64.vr,
                     sp.f64.vphi, sp.f64.vz, sp.f64.w, sp.f64.alive, sp.n, sp.n_cap, sp.chunked ? 1 : 0,
                     (uint32_t *)sp.f32.cell, sp.f32.fr, sp.f32.fz, sp.f32.vr, sp.f32.vphi, sp.f32.vz, sp.f32.w);
  return true;
}

void launch_f64_from_f32(Ctx &c, Species &sp) {
  if (sp.n <= 0 || !sp.f32.cell) return;
  hipLaunchKernelGGL(k_unpack, dim3(blocks_for(sp.n)), dim3(256), 0, c.stream, c.g, sp.f64.r, sp.f64.z,
                     sp.f64.vr, sp.f64.vphi, sp.f64.vz, sp.f64.w, sp.f64.alive, sp.n, sp.chunked ? 1 : 0,
                     (const uint32_t *)sp.f32.cell, sp.f32.fr, sp.f32.fz, sp.f32.vr, sp.f32.vphi, sp.f32.vz,
                     sp.f32.w);
}

// the work lists: one per tile shape that can be set (index into kTileShapes),
// and two whose tiles follow each species' size, for particles in cell order
// and in the ensemble sort's bands (kNumTiles, kNumTiles + 1)
constexpr int kEnsLists = kNumTiles + 2;
struct EnsParticles {
  int n_args = 0;
  F32Args *args = nullptr;
  GlobalSink *sinks = nullptr;
  EnsItem *items[kEnsLists] = {};
  int n_items[kEnsLists] = {};
};

namespace {
// a set shape's tiles are cut to one chunk for species below kSparsePpc
// particles per cell (a tile spans tile / ppc cells)
constexpr int kSparsePpc = 16;
// particles per lane (2^lg) of a species' tiles of 4 waves: the largest tile
// whose cells its boxes hold (the setting up of the boxes costs each tile the
// same, a particle past them gathers from HBM); unlike a single run's, an
// ensemble's tiles fill the GPU whatever their size.  In
// bands of two rows (species below 32 particles per cell, once the ensemble has
// sorted) a tile spans half as many columns.
int ens_auto_lg(const Ctx &c, const Species &sp, bool banded) {
  const double cells = (double)(c.g.nr - 1) * (double)(c.g.nz - 1);
  const double rows = banded && sp.n < 32 * cells ? 2 : 1;
  int lg = 4;
  while (lg > 0 && (256 << lg) * cells > rows * (kFK - 4) * (double)sp.n) lg--;
  return lg;
}
}  // namespace

int ens_lg(const Ctx &c, const Species &sp, int list) {
  if (list >= kNumTiles) return ens_auto_lg(c, sp, list == kNumTiles + 1);
  int lg = 0;
  while ((1 << lg) < kTileShapes[list][0]) lg++;
  if (sp.n < (long long)kSparsePpc * (c.g.nr - 1) * (c.g.nz - 1))
    while ((kTileShapes[list][1] * 64 << lg) > kChunk) lg--;
  return lg;
}

namespace {
std::vector<EnsItem> ens_list(const std::vector<Ctx *> &ctxs, int list) {
  std::vector<EnsItem> items, tiles;
  const int waves = list < kNumTiles ? kTileShapes[list][1] : kWavesPerBlock;
  int a = 0;
  for (Ctx *cp : ctxs) {
    Ctx &c = *cp;
    // every species by index, a bunch whether or not it has been created
    // (until its injection its particles are dead and do nothing)
    for (Species &sp : c.species) {
      if (sp.n_cap <= 0 || !sp.f32.cell) continue;
      if (!sp.chunked) {
        for (long long b = 0; b < sp.n_cap; b += waves * 64) items.push_back(EnsItem{a, -1, b, sp.n_cap});
      } else {
        const int lg = ens_lg(c, sp, list);
        const long long tile = (long long)waves * 64 << lg;
        for (long long t = 0; t * tile < sp.n_cap; t++) {
          // TileMap::base
          const long long per = tile < kChunk ? kChunk / tile : 1;
          const long long base = tile < kChunk ? t / per * kChunk + t % per * (tile / kPPT) : t * tile;
          tiles.push_back(EnsItem{a, lg, base, sp.n_cap});
        }
      }
      a++;
    }
  }
  items.insert(items.end(), tiles.begin(), tiles.end());
  return items;
}
}  // namespace

// the argument tables (a sort swaps the particle arrays); the work lists
// depend only on the species sizes and stay as built
int ens_particles_update(EnsParticles *e, const std::vector<Ctx *> &ctxs) {
  std::vector<F32Args> args;
  std::vector<GlobalSink> sinks;
  for (Ctx *cp : ctxs)
    for (int j = 0; j < (int)cp->species.size(); j++) {
      Species &sp = cp->species[j];
      if (sp.n_cap <= 0 || !sp.f32.cell) continue;
      args.push_back(args32(*cp, sp));
      sinks.push_back(sink32(*cp));
    }
  if ((int)args.size() != e->n_args) return -1;  // the species may not change
  if (hipMemcpy(e->args, args.data(), args.size() * sizeof(F32Args), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(e->sinks, sinks.data(), sinks.size() * sizeof(GlobalSink), hipMemcpyHostToDevice) != hipSuccess)
    return -1;
  return 0;
}

EnsParticles *ens_particles_build(const std::vector<Ctx *> &ctxs) {
  auto *e = new EnsParticles;
  for (Ctx *cp : ctxs)
    for (Species &sp : cp->species) e->n_args += sp.n_cap > 0 && sp.f32.cell ? 1 : 0;
  bool ok = hipMalloc((void **)&e->args, std::max(1, e->n_args) * sizeof(F32Args)) == hipSuccess &&
            hipMalloc((void **)&e->sinks, std::max(1, e->n_args) * sizeof(GlobalSink)) == hipSuccess;
  for (int t = 0; t < kEnsLists && ok; t++) {
    const std::vector<EnsItem> items = ens_list(ctxs, t);
    const size_t bytes = items.size() * sizeof(EnsItem);
    e->n_items[t] = (int)items.size();
    ok = hipMalloc((void **)&e->items[t], std::max(bytes, sizeof(EnsItem))) == hipSuccess &&
         (items.empty() || hipMemcpy(e->items[t], items.data(), bytes, hipMemcpyHostToDevice) == hipSuccess);
  }
  if (!ok || ens_particles_update(e, ctxs) != 0) {
    ens_particles_free(e);
    return nullptr;
  }
  return e;
}

int ens_auto_list(bool banded) { return kNumTiles + (banded ? 1 : 0); }

void ens_particles_free(EnsParticles *e) {
  if (!e) return;
  if (e->args) (void)hipFree(e->args);
  if (e->sinks) (void)hipFree(e->sinks);
  for (auto *p : e->items)
    if (p) (void)hipFree(p);
  delete e;
}

void ens_launch_inject(const EnsInjectItem *items, int n_items, int max_count, const long long *step,
                       hipStream_t st) {
  if (n_items <= 0 || max_count <= 0) return;
  const unsigned bx = (unsigned)std::min<long long>(((long long)max_count + 255) / 256, 4096);
  hipLaunchKernelGGL(k_ens_inject, dim3(bx, (unsigned)n_items), dim3(256), 0, st, items, step);
}

void ens_launch_count(long long *step, hipStream_t st) {
  hipLaunchKernelGGL(k_ens_count, dim3(1), dim3(64), 0, st, step);
}

void ens_launch_particles(EnsParticles *e, int list, hipStream_t st) {
  const int n = e->n_items[list], waves = list < kNumTiles ? kTileShapes[list][1] : kWavesPerBlock;
  if (n <= 0) return;
  auto kernel = waves == 4 ? k_ens_fused32<4> : waves == 2 ? k_ens_fused32<2> : k_ens_fused32<1>;
  hipLaunchKernelGGL(kernel, dim3(n), dim3(waves * 64), 0, st, e->args, e->sinks, e->items[list], n);
}

}  // namespace pdp3
