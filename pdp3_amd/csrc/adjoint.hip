// Hand-written adjoint of one loop iteration (src/loadInitParam.cpp:471-587)
// in the FP64 plain form's arithmetic, for gradients of a field objective with
// respect to the particle weights.
//
// Forward iteration n:  H^{n+1} = H^n + A E^n, Hh^n = H^n + A E^n / 2
//                       (x, v)^{n+1}, J^n = P((x, v)^n, E^n, Hh^n, w)
//                       E^{n+1} = Ke E^n - Kh (J^n - C H^{n+1})
// Backward, given the adjoints of E^{n+1}, H^{n+1} and the particle states:
//   1. lambda_J = -Kh lambda_E;  lambda_H += C^T (Kh lambda_E);  lambda_E <- Ke lambda_E
//   2. per particle, the vector-Jacobian product of P, written out in reverse:
//      every output (new r, z, v and each grid deposit) passes its adjoint back
//      to the 12 inputs (r, z, v, the gathered E and H, w); the adjoints of the
//      gathered fields are scattered to the nodes with the gather weights, the
//      weight adjoint is accumulated per particle
//   3. lambda_alpha = lambda_H + lambda_Hh / 2;  lambda_E += A^T lambda_alpha;
//      lambda_H <- lambda_H + lambda_Hh
// The operators A (HField::calc_field, src/hField.cpp:93-157), C, Ke, Kh
// (EField::calc_field, src/eField.cpp:85-170, PML in Ke / Kh) are transposed
// node by node in pull form (no atomics).
#include <algorithm>
#include <climits>
#include <type_traits>

#include "context.hpp"
#include "crmath.hpp"
#include "sink.hpp"

namespace pdp3 {

namespace {

constexpr int kDN = 4;  // directions
static_assert(kDN == kTangentDirs, "the tangent-linear model runs kDN directions");

// dual numbers of kDN directions (strict_d, whose four inputs they are)
struct D {
  double v;
  double d[kDN];
};

__device__ __forceinline__ D cst(double x) {
  D r;
  r.v = x;
  for (int j = 0; j < kDN; j++) r.d[j] = 0.0;
  return r;
}
// x as direction `dir` (derivative 1 there); selects on constant indices, so
// that no dual number is addressed through memory
__device__ __forceinline__ D seed(double x, int dir) {
  D r;
  r.v = x;
#pragma unroll
  for (int j = 0; j < kDN; j++) r.d[j] = j == dir ? 1.0 : 0.0;
  return r;
}
__device__ __forceinline__ D operator+(D a, D b) {
  D r;
  r.v = a.v + b.v;
  for (int j = 0; j < kDN; j++) r.d[j] = a.d[j] + b.d[j];
  return r;
}
__device__ __forceinline__ D operator-(D a, D b) {
  D r;
  r.v = a.v - b.v;
  for (int j = 0; j < kDN; j++) r.d[j] = a.d[j] - b.d[j];
  return r;
}
__device__ __forceinline__ D operator-(D a) {
  D r;
  r.v = -a.v;
  for (int j = 0; j < kDN; j++) r.d[j] = -a.d[j];
  return r;
}
__device__ __forceinline__ D operator*(D a, D b) {
  D r;
  r.v = a.v * b.v;
  for (int j = 0; j < kDN; j++) r.d[j] = a.d[j] * b.v + a.v * b.d[j];
  return r;
}
__device__ __forceinline__ D operator/(D a, D b) {
  D r;
  r.v = a.v / b.v;
  const double ib = 1.0 / b.v;
  for (int j = 0; j < kDN; j++) r.d[j] = (a.d[j] - r.v * b.d[j]) * ib;
  return r;
}
__device__ __forceinline__ D operator+(D a, double b) { return a + cst(b); }
__device__ __forceinline__ D operator+(double a, D b) { return cst(a) + b; }
__device__ __forceinline__ D operator-(D a, double b) { return a - cst(b); }
__device__ __forceinline__ D operator-(double a, D b) { return cst(a) - b; }
__device__ __forceinline__ D operator*(D a, double b) {
  D r;
  r.v = a.v * b;
  for (int j = 0; j < kDN; j++) r.d[j] = a.d[j] * b;
  return r;
}
__device__ __forceinline__ D operator*(double a, D b) {
  D r;
  r.v = a * b.v;
  for (int j = 0; j < kDN; j++) r.d[j] = a * b.d[j];
  return r;
}
__device__ __forceinline__ D operator/(D a, double b) {
  D r;
  r.v = a.v / b;
  for (int j = 0; j < kDN; j++) r.d[j] = a.d[j] / b;
  return r;
}
__device__ __forceinline__ D operator/(double a, D b) { return cst(a) / b; }
constexpr double kC2 = kLightSpeed * kLightSpeed;

// ------------------------------------------------------------ the particle

struct AdjFields {
  const double *er, *ephi, *ez, *hhr, *hhphi, *hhz;  // E^n, Hh^n
};
struct AdjGrid {
  const double *ljr, *ljphi, *ljz;             // adjoint of J^n
  double *ler, *lephi, *lez, *lhr, *lhphi, *lhz;  // adjoint of E^n, Hh^n (scatter, atomics)
};
// what a species' charge, mass and the grid's constants come to: the scales of
// the push's E and H (q / m does not depend on the weight), and of the deposits
// of one charge into J_z, J_r and J_phi
struct StepScales {
  double es, bs, kz, kr, kj;
};
StepScales scales_of(const GridDesc &g, double q, double m, bool vay) {
  const double c1 = q * g.dt / (2 * m);
  return StepScales{vay ? 2 * c1 : c1, vay ? kMagnConst * c1 * (2 * c1) * c1 : kMagnConst * c1,
                    q / (4.0 * kPi * g.dr * g.dr * g.dt), q / (2.0 * kPi * g.dr * g.dz * g.dt), q / (2.0 * g.dz * g.dr)};
}
struct AdjSpecies {
  StateRef st;                          // state at step n
  double *lr, *lz, *lvr, *lvphi, *lvz;  // in: adjoint of the state after step n; out: before
  double *lw;                           // accumulated adjoint of the weight
  double charge;
  StepScales k;
  long long n;                          // slots
};

// the particle in slot i of either form, in FP64 as a download gives it (r and
// z from the cell and its offsets, v = u / gamma in the FP32 form); false: dead
struct AdjParticle {
  double r, z, vr, vphi, vz, w;
};
template <bool F32>
__device__ __forceinline__ bool adj_load(const GridDesc &g, const StateRef &s, long long i, AdjParticle &p) {
  if (F32) {
    const uint32_t c = s.cell[i];
    if (c & 0x80000000u) return false;
    p.r = ((double)(int)((c >> 16) & 0x7FFF) + (double)s.fa[i]) * g.dr;
    p.z = ((double)(int)(c & 0xFFFF) + (double)s.fb[i]) * g.dz;
    const double u0 = s.ur[i], u1 = s.uphi[i], u2 = s.uz[i];
    const double ig = 1.0 / sqrt(1.0 + (u0 * u0 + u1 * u1 + u2 * u2) / (kLightSpeed * kLightSpeed));
    p.vr = u0 * ig;
    p.vphi = u1 * ig;
    p.vz = u2 * ig;
    p.w = s.fw[i];
  } else {
    if (s.alive[i] != 1) return false;
    p.r = s.r[i];
    p.z = s.z[i];
    p.vr = s.vr[i];
    p.vphi = s.vphi[i];
    p.vz = s.vz[i];
    p.w = s.w[i];
  }
  return true;
}
// the slot of this thread: plasma blocks take 256 consecutive logical
// particles of the chunked layout, which lie along one run of cells
template <bool BUNCH>
__device__ __forceinline__ long long adj_slot() {
  if (BUNCH) return (long long)blockIdx.x * blockDim.x + threadIdx.x;
  return TileMap<1, 4>::base(blockIdx.x) + TileMap<1, 4>::first(threadIdx.x);
}

// node of box[.][0][0] of kR x kK nodes, from the thread's cell (INT_MAX: dead): a bunch
// block's boxes begin one row and two columns below its smallest cell, a plasma
// block's lie around its median cell.  (After a barrier, which the cleared box
// needs too.)
template <bool BUNCH, int kR, int kK>
__device__ __forceinline__ void block_anchor(int &i, int &k, bool live) {
  if (BUNCH) {
    block_min2(i, k);
    if (i == INT_MAX) i = k = 0;
    i -= 1;
    k -= 2;
  } else {
    block_median(i, k, live);
    i -= kR / 2 - 1;
    k -= kK / 2 - 1;
  }
}

// quotients by the context's constants and row volumes take their reciprocals
// from the context (div_cr: correctly rounded, as the IEEE division): a quotient
// is five FP64 operations instead of eleven and a quarter-rate reciprocal, and the
// particle steps, bound by their instructions at two waves per SIMD (211 VGPRs; three
// spill 40 and take 290 us; the reverse step 1743 vector instructions a particle, 976
// of them FP64), had about fifty of them: reverse step of 2.6e6 particles 238 us with
// the IEEE quotients, 213 us
__device__ __forceinline__ double per_dr(const GridDesc &g, double x) { return div_cr(x, g.dr, g.inv_dr); }
__device__ __forceinline__ double per_dz(const GridDesc &g, double x) { return div_cr(x, g.dz, g.inv_dz); }
__device__ __forceinline__ double per_c2(double x) { return div_cr(x, kC2, 1.0 / kC2); }
__device__ __forceinline__ int cell_r(const GridDesc &g, double r) { return (int)ceil(per_dr(g, r)) - 1; }
__device__ __forceinline__ int cell_z(const GridDesc &g, double z) { return (int)ceil(per_dz(g, z)) - 1; }
// {volume, 1 / volume} of row i's cells (a row outside the grid is kept inside
// the table; it receives and holds nothing), and of the axis cell
__device__ __forceinline__ double2 vol_row(const GridDesc &g, int i) { return g.vol[min(i, g.nr + 1)]; }
__device__ __forceinline__ double2 vol_axis(const GridDesc &g) { return make_double2(g.cyl, g.inv_cyl); }

constexpr int kAR = 0, kAPhi = 1, kAZ = 2;

// strict_motion_weighting, src/particles.cpp:786-988
template <class S>
__device__ void strict_d(const GridDesc &g, S &acc, D q, D radius_new, D longitude_new, D radius_old,
                         D longitude_old) {
  const double dr = g.dr, dz = g.dz, delta_t = g.dt;
  int i_n = cell_r(g, radius_new.v), k_n = cell_z(g, longitude_new.v);
  int i_o = cell_r(g, radius_old.v), k_o = cell_z(g, longitude_old.v);
  if (i_n < 0) i_n = 0;
  if (k_n < 0) k_n = 0;
  if (i_o < 0) i_o = 0;
  if (k_o < 0) k_o = 0;
  bool still_r = fabs(radius_new.v - radius_old.v) < kMnzl;
  bool still_z = fabs(longitude_new.v - longitude_old.v) < kMnzl;
  if (still_r && still_z) return;
  if (still_r) {
    D value_part = 2. * kPi * radius_new * dr * dz;
    D r1 = radius_new - 0.5 * dr, r3 = radius_new + 0.5 * dr;
    D r2 = cst((i_n + 0.5) * dr);
    D wl, wu;
    if (i_n == 0)
      wl = q / (delta_t * kPi * dr * dr / 4.) * kPi * (r2 * r2 - r1 * r1) / value_part;
    else
      wl = q / (delta_t * 2. * kPi * i_n * dr * dr) * kPi * (r2 * r2 - r1 * r1) / value_part;
    wu = q / (delta_t * 2 * kPi * (i_n + 1) * dr * dr) * kPi * (r3 * r3 - r2 * r2) / value_part;
    int res_k = k_n - k_o;
    if (res_k == 0) {
      D delta_z = longitude_new - longitude_old;
      acc.add(kAZ, i_n, k_n, wl * delta_z);
      acc.add(kAZ, i_n + 1, k_n, wu * delta_z);
    } else if (res_k == 1) {
      D delta_z = k_n * dz - longitude_old;
      acc.add(kAZ, i_n, k_n - 1, wl * delta_z);
      acc.add(kAZ, i_n + 1, k_n - 1, wu * delta_z);
      delta_z = longitude_new - k_n * dz;
      acc.add(kAZ, i_n, k_n, wl * delta_z);
      acc.add(kAZ, i_n + 1, k_n, wu * delta_z);
    } else if (res_k == -1) {
      D delta_z = (k_n + 1) * dz - longitude_old;
      acc.add(kAZ, i_n, k_n + 1, wl * delta_z);
      acc.add(kAZ, i_n + 1, k_n + 1, wu * delta_z);
      delta_z = longitude_new - (k_n + 1) * dz;
      acc.add(kAZ, i_n, k_n, wl * delta_z);
      acc.add(kAZ, i_n + 1, k_n, wu * delta_z);
    }
  } else if (still_z) {
    int res_i = i_n - i_o;
    D left_delta_z = (k_n + 1) * dz - longitude_new;
    D right_delta_z = longitude_new - k_n * dz;
    auto part = [&](D delta_r, double r0, D rad_old) {
      D ssd = q / (kPi * 4. * r0 * dz * dz * dr * delta_t);
      return ssd * (delta_r - r0 * r0 / (rad_old + delta_r) + r0 * r0 / rad_old + dr * dr / (4. * (rad_old + delta_r)) -
                    dr * dr / (4. * rad_old));
    };
    if (res_i == 0) {
      D wj = part(radius_new - radius_old, (i_n + 0.5) * dr, radius_old);
      acc.add(kAR, i_n, k_n, wj * left_delta_z);
      acc.add(kAR, i_n, k_n + 1, wj * right_delta_z);
    } else if (res_i == 1) {
      D wj = part(i_n * dr - radius_old, (i_n - 0.5) * dr, radius_old);
      acc.add(kAR, i_n - 1, k_n, wj * left_delta_z);
      acc.add(kAR, i_n - 1, k_n + 1, wj * right_delta_z);
      // the reference's `r0 * r0 / i_n * dr` (src/particles.cpp:941)
      D delta_r = radius_new - i_n * dr;
      const double r0 = (i_n + 0.5) * dr;
      D ssd = q / (kPi * 4. * r0 * dz * dz * dr * delta_t);
      wj = ssd * (delta_r - r0 * r0 / (i_n * dr + delta_r) + r0 * r0 / i_n * dr + dr * dr / (4. * (i_n * dr + delta_r)) -
                  dr * dr / (4. * i_n * dr));
      acc.add(kAR, i_n, k_n, wj * left_delta_z);
      acc.add(kAR, i_n, k_n + 1, wj * right_delta_z);
    } else if (res_i == -1) {
      D wj = part((i_n + 1) * dr - radius_old, (i_n + 1.5) * dr, radius_old);
      acc.add(kAR, i_n + 1, k_n, wj * left_delta_z);
      acc.add(kAR, i_n + 1, k_n + 1, wj * right_delta_z);
      D delta_r = radius_new - (i_n + 1) * dr;
      const double r0 = (i_n + 0.5) * dr;
      D ssd = q / (kPi * 4. * r0 * dz * dz * dr * delta_t);
      wj = ssd * (delta_r - r0 * r0 / ((i_n + 1) * dr + delta_r) + r0 * r0 / (i_n + 1) * dr +
                  dr * dr / (4. * ((i_n + 1) * dr + delta_r)) - dr * dr / (4. * (i_n + 1) * dr));
      acc.add(kAR, i_n, k_n, wj * left_delta_z);
      acc.add(kAR, i_n, k_n + 1, wj * right_delta_z);
    }
  }
}

// ------------------------------------------------ reverse mode, one particle
#pragma clang fp contract(fast)
// The vector-Jacobian product of one particle's step, written out stage by
// stage in reverse.  Every deposit is linear in the weight and the push does
// not depend on it (q / m), so the weight's adjoint is the sum of lambda_J
// times the deposits of a unit weight.  One forward evaluation and one reverse sweep
// replace 12 directional derivatives of the step.

struct V3 {
  double x, y, z;
};
__device__ __forceinline__ V3 operator+(V3 a, V3 b) { return V3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ V3 operator*(double s, V3 a) { return V3{s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 cross(V3 a, V3 b) {
  return V3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ V3 fma3(double s, V3 a, V3 b) { return V3{s * a.x + b.x, s * a.y + b.y, s * a.z + b.z}; }

// u = v gamma(v) and gamma = (1 + u^2/c^2)^(-1/2) with their reverse steps
struct Boost {
  V3 u;       // v with the components below MNZL dropped
  double g0;  // 1 / sqrt(1 - v^2/c^2)
};
__device__ __forceinline__ Boost boost_of(V3 v) {
  Boost b;
  b.u = V3{fabs(v.x) < kMnzl ? 0.0 : v.x, fabs(v.y) < kMnzl ? 0.0 : v.y, fabs(v.z) < kMnzl ? 0.0 : v.z};
  b.g0 = rsqrt_near(1.0 - per_c2(dot(b.u, b.u)));
  return b;
}
// adjoint of v from the adjoint of U = g0 u
__device__ __forceinline__ V3 boost_back(const Boost &b, V3 v, V3 lU) {
  const double s = per_c2(b.g0 * b.g0 * b.g0) * dot(lU, b.u);
  const V3 l = fma3(s, b.u, b.g0 * lU);
  return V3{fabs(v.x) < kMnzl ? 0.0 : l.x, fabs(v.y) < kMnzl ? 0.0 : l.y, fabs(v.z) < kMnzl ? 0.0 : l.z};
}
__device__ __forceinline__ double inv_gamma(V3 u) { return rsqrt_near(1.0 + per_c2(dot(u, u))); }
// adjoint of u added for an adjoint lg of g = inv_gamma(u)
__device__ __forceinline__ V3 inv_gamma_back(double g, V3 u, double lg, V3 l) {
  return fma3(per_c2(-(g * g * g)) * lg, u, l);
}

// what the reverse sweep of a push keeps of its forward evaluation, recomputed
// from the inputs: v, and the fields multiplied by the species' scales
struct PushBack {
  V3 v, e, b;  // adjoints of v and of the scaled fields
};

// relativistic Boris (src/particles.cpp:1025-1150)
__device__ __forceinline__ V3 boris_fwd(V3 v, V3 e, V3 h) {
  const Boost b0 = boost_of(v);
  const V3 t = fma3(b0.g0, b0.u, e);
  const V3 b = inv_gamma(t) * h;
  const V3 w = cross(t + cross(t, b), b);
  const V3 u = fma3(2.0 / (1.0 + dot(b, b)), w, t) + e;
  return inv_gamma(u) * u;
}
__device__ __forceinline__ PushBack boris_back(V3 v, V3 e, V3 h, V3 lv) {
  const Boost b0 = boost_of(v);
  const V3 t = fma3(b0.g0, b0.u, e);
  const double g1 = inv_gamma(t);
  const V3 b = g1 * h;
  const V3 tp = t + cross(t, b);
  const double c2 = 2.0 / (1.0 + dot(b, b));
  const V3 w = cross(tp, b);
  const V3 u = fma3(c2, w, t) + e;
  const double g2 = inv_gamma(u);
  PushBack o;
  const V3 lu = inv_gamma_back(g2, u, dot(lv, u), g2 * lv);
  const double lc2 = dot(lu, w);
  const V3 lw = c2 * lu;
  const V3 ltp = cross(b, lw);
  V3 lt = lu + ltp + cross(b, ltp);
  V3 lb = cross(lw, tp) + cross(ltp, t);
  lb = fma3(-c2 * c2 * lc2, b, lb);
  o.b = g1 * lb;
  lt = inv_gamma_back(g1, t, dot(lb, h), lt);
  o.e = lu + lt;
  o.v = boost_back(b0, v, lt);
  return o;
}

// Vay with the reference's scaling (src/particles.cpp:1152-1254)
__device__ __forceinline__ V3 vay_fwd(V3 v, V3 e, V3 h) {
  const Boost b0 = boost_of(v);
  const V3 t = b0.g0 * b0.u;
  const V3 up = fma3(inv_gamma(t), cross(t, h), t + e);
  const double B2 = dot(h, h), ub = dot(up, h), sg = 1.0 + per_c2(dot(up, up)) - B2;
  const double al = rsqrt_near(0.5 * (sg + sqrt(sg * sg + 4. * (B2 + ub * ub))));
  const V3 b = al * h;
  const V3 u = (1.0 / (1.0 + dot(b, b))) * (fma3(dot(up, b), b, up) + cross(up, b));
  return inv_gamma(u) * u;
}
__device__ __forceinline__ PushBack vay_back(V3 v, V3 e, V3 h, V3 lv) {
  const Boost b0 = boost_of(v);
  const V3 t = b0.g0 * b0.u;
  const double g1 = inv_gamma(t);
  const V3 th = cross(t, h);
  const V3 up = fma3(g1, th, t + e);
  const double B2 = dot(h, h), ub = dot(up, h), sg = 1.0 + per_c2(dot(up, up)) - B2;
  const double root = sqrt(sg * sg + 4. * (B2 + ub * ub));
  const double al = rsqrt_near(0.5 * (sg + root));
  const V3 b = al * h;
  const double s = 1.0 / (1.0 + dot(b, b)), al2 = dot(up, b);
  const V3 q = fma3(al2, b, up) + cross(up, b);
  const V3 u = s * q;
  const double g3 = inv_gamma(u);
  PushBack o;
  const V3 lu = inv_gamma_back(g3, u, dot(lv, u), g3 * lv);
  const double ls = dot(lu, q);
  const V3 lq = s * lu;
  const double lal2 = dot(lq, b);
  V3 lup = fma3(lal2, b, lq + cross(b, lq));
  V3 lb = fma3(lal2, up, fma3(al2, lq, cross(lq, up)));
  lb = fma3(-2.0 * s * s * ls, b, lb);
  const double lx = -0.5 * al * al * al * dot(lb, h);
  const double lin = 0.5 * lx * 0.5 / root;
  const double lsg = 0.5 * lx + 2.0 * sg * lin, lub = 2.0 * ub * 4.0 * lin, lB2 = 4.0 * lin - lsg;
  lup = fma3(lub, h, fma3(lsg * (2.0 / kC2), up, lup));
  V3 lh = fma3(al, lb, fma3(lub, up, (2.0 * lB2) * h));
  const V3 mu = g1 * lup;
  lh = lh + cross(mu, t);
  const V3 lt = inv_gamma_back(g1, t, dot(lup, th), cross(h, mu));
  o.e = lup;
  o.b = lh;
  o.v = boost_back(b0, v, lup + lt);
  return o;
}

// the four-node gather of one component and its derivatives along r and z
// (src/eField.cpp:204-316), from the shares of the rings (per unit of z) of
// its radial family
struct RingW {
  int ir;
  double in, out, din, dout;  // shares of nodes ir, ir+1 and their r derivatives
};
__device__ __forceinline__ RingW ring_lo(const GridDesc &g, double r) {
  RingW w;
  w.ir = min(max(cell_r(g, r - 0.5 * g.dr), 0), g.nr - 2);
  const double r1 = r - 0.5 * g.dr, r3 = r + 0.5 * g.dr, r2 = (w.ir + 1) * g.dr;
  const double2 v1 = vol_row(g, w.ir + 1), v2 = vol_row(g, w.ir + 3);
  const double p1 = div_cr(kPi, v1.x, v1.y), p2 = div_cr(kPi, v2.x, v2.y);
  w.in = p1 * (r2 * r2 - r1 * r1);
  w.out = p2 * (r3 * r3 - r2 * r2);
  w.din = -2.0 * p1 * r1;
  w.dout = 2.0 * p2 * r3;
  return w;
}
__device__ __forceinline__ RingW ring_own(const GridDesc &g, double r) {
  RingW w;
  w.ir = min(max(cell_r(g, r), 0), g.nr - 2);
  const double r1 = r - 0.5 * g.dr, r3 = r + 0.5 * g.dr, r2 = (w.ir + 0.5) * g.dr;
  const double2 v1 = (r > g.dr) ? vol_row(g, w.ir) : vol_axis(g), v2 = vol_row(g, w.ir + 2);
  const double p1 = div_cr(kPi, v1.x, v1.y), p2 = div_cr(kPi, v2.x, v2.y);
  w.in = p1 * (r2 * r2 - r1 * r1);
  w.out = p2 * (r3 * r3 - r2 * r2);
  w.din = -2.0 * p1 * r1;
  w.dout = 2.0 * p2 * r3;
  return w;
}
struct ColW {
  int kz;
  double d1, d2;  // distances to column kz+1 and from column kz
};
__device__ __forceinline__ ColW col_w(const GridDesc &g, double z, bool half) {
  ColW c;
  c.kz = min(max(cell_z(g, half ? z - 0.5 * g.dz : z), 0), g.nz - 2);
  const double z0 = (half ? c.kz + 0.5 : c.kz) * g.dz;
  c.d1 = z0 + g.dz - z;
  c.d2 = z - z0;
  return c;
}
struct Gathered {
  double v, dr, dz;
};
__device__ __forceinline__ Gathered gather_grad(const GridDesc &g, const double *F, const RingW &w, const ColW &c) {
  const double *row0 = F + (size_t)w.ir * (size_t)g.nz + c.kz;
  const double *row1 = row0 + g.nz;
  const double f00 = row0[0], f01 = row0[1], f10 = row1[0], f11 = row1[1];
  const double lo = f00 * c.d1 + f01 * c.d2, hi = f10 * c.d1 + f11 * c.d2;
  return Gathered{w.in * lo + w.out * hi, w.din * lo + w.dout * hi, w.in * (f01 - f00) + w.out * (f11 - f10)};
}

// the adjoints of the gathered fields of one block's particles are summed in
// an LDS box of kR x kABK nodes per component (block_anchor) and added to the
// grid once per block; stencils outside the box go to the grid directly.  A plasma
// block lies along one row.  A bunch block spans the bunch's radius: in four rows
// most of its 24 atomics a particle went to the same few grid nodes, and 6.4e4
// bunch particles took as long as 2.6e6 plasma particles (330 us).
constexpr int kABK = 64, kABComp = 6;
template <bool BUNCH>
struct AdjBox {
  static constexpr bool kBunch = BUNCH;
  static constexpr int kR = BUNCH ? 16 : 4;
  double *box;  // LDS, kABComp x kR x kABK
  int bi, bk;   // node of box[.][0][0]
};
template <class Box>
__device__ __forceinline__ void box_scatter(const GridDesc &g, const Box &b, int comp, double *LF, const RingW &w,
                                            const ColW &c, double lam) {
  if (lam == 0.0) return;
  // the shares of the nodes (ir, kz), (ir+1, kz), (ir, kz+1), (ir+1, kz+1)
  const double v00 = w.in * c.d1 * lam, v10 = w.out * c.d1 * lam, v01 = w.in * c.d2 * lam, v11 = w.out * c.d2 * lam;
  const int li = w.ir - b.bi, lk = c.kz - b.bk;
  if ((unsigned)li < (unsigned)(Box::kR - 1) && (unsigned)lk < (unsigned)(kABK - 1)) {
    double *q = b.box + (comp * Box::kR + li) * kABK + lk;
    atomicAdd(q, v00);
    atomicAdd(q + kABK, v10);
    atomicAdd(q + 1, v01);
    atomicAdd(q + kABK + 1, v11);
  } else {
    double *row0 = LF + (size_t)w.ir * (size_t)g.nz + c.kz;
    double *row1 = row0 + g.nz;
    unsafeAtomicAdd(row0, v00);
    unsafeAtomicAdd(row1, v10);
    unsafeAtomicAdd(row0 + 1, v01);
    unsafeAtomicAdd(row1 + 1, v11);
  }
}

// lambda_J at node (i, k), 0 off the grid
__device__ __forceinline__ double lam_at(const GridDesc &g, const double *L, int i, int k) {
  if ((unsigned)i >= (unsigned)g.nr || (unsigned)k >= (unsigned)g.nz) return 0.0;
  return L[(size_t)i * (size_t)g.nz + (size_t)k];
}

// reverse of the J_phi deposit (azimuthal_current_distribution,
// src/particles.cpp:688-784) of w charges q: adds to the adjoints of r, z,
// v_phi; returns the weight's, sum lambda_J J / w
__device__ __forceinline__ double jphi_back(const GridDesc &g, const double *L, double kj, double w, double r, double z,
                                            double vphi, double &lr, double &lz, double &lvphi) {
  const double dr = g.dr, dz = g.dz;
  const int i = max(cell_r(g, r), 0), k = max(cell_z(g, z), 0);
  const double r1 = r - 0.5 * dr, r2 = (i + 0.5) * dr, r3 = r + 0.5 * dr;
  const double i1 = (r > dr) ? vol_row(g, i).y : g.inv_cyl, i2 = vol_row(g, i + 1).y;
  const double d1 = (k + 0.5) * dz - (z - 0.5 * dz), d2 = (z + 0.5 * dz) - (k + 0.5) * dz;
  const double l00 = lam_at(g, L, i, k) * i1, l10 = lam_at(g, L, i + 1, k) * i2;
  const double l01 = lam_at(g, L, i, k + 1) * i1, l11 = lam_at(g, L, i + 1, k + 1) * i2;
  const double in = r2 * r2 - r1 * r1, out = r3 * r3 - r2 * r2;
  const double lo = l00 * d1 + l01 * d2, hi = l10 * d1 + l11 * d2;
  const double G = in * lo + out * hi;
  const double ir = 1.0 / r, K = kj * ir;
  lvphi += w * K * G;
  lr += w * K * vphi * (2.0 * (r3 * hi - r1 * lo) - G * ir);
  lz += w * K * vphi * (in * (l01 - l00) + out * (l11 - l10));
  return K * vphi * G;
}

// M(x) = (log(1+x) - x) / x and its derivative (series below |x| = 0.1)
__device__ __forceinline__ void m_and_slope(double x, double &M, double &dM) {
  if (fabs(x) < 0.1) {
    const double c[] = {1.0 / 11.0, -0.1, 1.0 / 9.0, -0.125, 1.0 / 7.0, -1.0 / 6.0, 0.2, -0.25, 1.0 / 3.0, -0.5};
    double s = -1.0 / 12.0, d = 0.0;
    for (double ck : c) {
      d = s + x * d;
      s = ck + x * s;
    }
    M = x * s;
    dM = s + x * d;
  } else {
    M = (log1p(x) - x) / x;
    dM = (1.0 / (1.0 + x) - 1.0 - M) / x;
  }
}

// The deposits of one straight piece inside cell (i, k)
// (simple_current_distribution, src/particles.cpp:333-474), as integrals written
// without cancellation in cell units (r = (i + a) dr, z = (k + b) dz, rho = i + a,
// rho_e = rho + drho, x = drho / rho, M = (ln(1+x) - x) / x, N = -x / (1+x) - M):
//   J_z[i]   = q dzeta / (4 pi dr^2 dt) [ (1-a)(2i+a)/rho - drho/2 + i(i+1)/rho M ] / i
//   J_z[i+1] = q dzeta / (4 pi dr^2 dt) [ a(2i+1+a)/rho + drho/2 - i(i+1)/rho M ] / (i+1)
//   J_r[k]   = q / (2 pi dr dz dt) [ drho((1-b)/2 - dzeta/4) + i(i+1)/(2 rho) (drho (1-b)/rho_e + dzeta N) ] / (i+1/2)
//   J_r[k+1] = q / (2 pi dr dz dt) [ drho(b/2 + dzeta/4) + i(i+1)/(2 rho) (drho b/rho_e - dzeta N) ] / (i+1/2)
// (and the polynomial forms on the axis cell).  The reference's forms are
// differences of O(i) terms: their derivative loses ~1/x digits for nearly
// axial paths, which a relativistic beam's particles are.
//
// Reverse of one piece: S = sum lambda_J J and its derivatives with respect to
// the piece's ends.
struct PieceAdj {
  double s, rn, zn, ro, zo;
};
__device__ __forceinline__ PieceAdj segment_back(const GridDesc &g, const AdjGrid &lg, const StepScales &s, double rn, double zn,
                                                 double ro, double zo, int i, int k) {
  const double dr = g.dr, dz = g.dz;
  PieceAdj o{0.0, 0.0, 0.0, 0.0, 0.0};
  if ((fabs(rn - ro) < kMnzl) || (fabs(zn - zo) < kMnzl)) return o;
  const double fi = (double)i;
  const double a = per_dr(g, ro) - fi, b = per_dz(g, zo) - (double)k;
  const double drho = per_dr(g, rn - ro), dzeta = per_dz(g, zn - zo);
  // lambda_J times the scales of the pairs (without the dzeta of J_z)
  double gz0 = s.kz * lam_at(g, lg.ljz, i, k), gz1 = s.kz * lam_at(g, lg.ljz, i + 1, k);
  double gr0 = s.kr * lam_at(g, lg.ljr, i, k), gr1 = s.kr * lam_at(g, lg.ljr, i, k + 1);
  const double hdr = 0.5 * drho, ub = 1.0 - b, qdz = 0.25 * dzeta;
  double sa, sb, sdr, sdz;
  if (i == 0) {
    const double j0 = 8.0 * (1.0 - hdr - a), j1 = hdr + 1.0 + a;
    gr0 *= 2.0;
    gr1 *= 2.0;
    const double p0 = 0.5 * ub - qdz, p1 = 0.5 * b + qdz;
    sdz = gz0 * j0 + gz1 * j1;
    o.s = dzeta * sdz + drho * (gr0 * p0 + gr1 * p1);
    sa = dzeta * (gz1 - 8.0 * gz0);
    sdr = dzeta * (0.5 * gz1 - 4.0 * gz0) + gr0 * p0 + gr1 * p1;
    sb = 0.5 * drho * (gr1 - gr0);
    sdz += 0.25 * drho * (gr1 - gr0);
  } else {
    gz0 /= fi;
    gz1 /= fi + 1.0;
    const double ih = 1.0 / (fi + 0.5);
    gr0 *= ih;
    gr1 *= ih;
    const double rs = fi + a, re = rs + drho, irs = 1.0 / rs, ire = 1.0 / re;
    const double ii = fi * (fi + 1.0), x = drho * irs, t = drho * ire;
    double M, dM;
    m_and_slope(x, M, dM);
    const double N = -t - M, iiM = ii * M, cc = 0.5 * ii * irs;
    const double A0 = (1.0 - a) * (2.0 * fi + a) + iiM, A1 = a * (2.0 * fi + 1.0 + a) - iiM;
    const double R0 = t * ub + dzeta * N, R1 = t * b - dzeta * N;
    const double p0 = 0.5 * ub - qdz, p1 = 0.5 * b + qdz;
    const double gd = gr0 - gr1;
    const double jz = gz0 * (A0 * irs - hdr) + gz1 * (A1 * irs + hdr);  // per unit of dzeta
    const double grR = gr0 * R0 + gr1 * R1, grp = gr0 * p0 + gr1 * p1;
    o.s = dzeta * jz + drho * grp + cc * grR;
    sdz = jz + gd * (cc * N - 0.25 * drho);
    sb = -gd * (hdr + cc * t);
    const double sM = dzeta * (gz0 - gz1) * ii * irs - gd * cc * dzeta;
    const double st = cc * (gr0 * ub + gr1 * b - dzeta * gd);
    const double sirs = dzeta * (gz0 * A0 + gz1 * A1) + 0.5 * ii * grR;
    const double sx = sM * dM;
    sa = dzeta * irs * (gz0 * (1.0 - 2.0 * fi - 2.0 * a) + gz1 * (2.0 * fi + 1.0 + 2.0 * a)) - sirs * irs * irs -
         sx * x * irs - st * t * ire;
    sdr = 0.5 * dzeta * (gz1 - gz0) + grp + sx * irs + st * rs * ire * ire;
  }
  o.rn = sdr * g.inv_dr;
  o.ro = (sa - sdr) * g.inv_dr;
  o.zn = sdz * g.inv_dz;
  o.zo = (sb - sdz) * g.inv_dz;
  return o;
}

// strict_d's sink in the reverse sweep: its four inputs are the dual
// directions, the deposits are linear in q
struct StrictSink {
  const GridDesc *g;
  const AdjGrid *lg;
  PieceAdj o;
  __device__ __forceinline__ void add(int comp, int i, int k, D v) {
    const double l = lam_at(*g, comp == kAR ? lg->ljr : lg->ljz, i, k);
    o.s += l * v.v;
    o.rn += l * v.d[0];
    o.zn += l * v.d[1];
    o.ro += l * v.d[2];
    o.zo += l * v.d[3];
  }
};

// the straight path (ro, zo) -> (rn, zn) (current_distribution,
// src/particles.cpp:480-685): its ns pieces, split at the radial face r = rb
// (met at z1) and the axial face z = zb (met at r2) that it crosses, rfirst: in
// that order; the last piece lies in cell (i_n, k_n), those before it in
// (i0, k0) and (i1, k1)
struct Path {
  int i_n, k_n, i0, k0, i1, k1, ns;
  bool strict, rad, axi, rfirst;  // strict: along one axis, not split
  double rb, zb, z1, r2, slope;
};
__device__ __forceinline__ Path split_path(const GridDesc &g, double rn, double zn, double ro, double zo) {
  const double dr = g.dr, dz = g.dz;
  Path p;
  int i_n = max(cell_r(g, rn), 0), k_n = max(cell_z(g, zn), 0);
  int i_o = max(cell_r(g, ro), 0), k_o = max(cell_z(g, zo), 0);
  if (ro == (i_o + 1) * dr) i_o = i_n;
  if (zo == (k_o + 1) * dz) k_o = k_n;
  if (rn == (i_n + 1) * dr) i_n = i_o;
  if (zn == (k_n + 1) * dz) k_n = k_o;
  const int di = i_n - i_o, dk = k_n - k_o, res = abs(di) + abs(dk);
  p.strict = (fabs(rn - ro) < kMnzl) || (fabs(zn - zo) < kMnzl);
  p.ns = 1;
  p.i_n = p.i0 = p.i1 = i_n;
  p.k_n = p.k0 = p.k1 = k_n;
  p.rad = p.axi = p.rfirst = false;
  p.rb = p.zb = p.z1 = p.r2 = 0.0;
  p.slope = (rn - ro) / (zn - zo);
  if (res == 1) {
    p.ns = 2;
    if (di != 0) {
      p.rad = p.rfirst = true;
      const bool up = !(ro > (i_n + 1) * dr);
      p.rb = (up ? i_n : i_n + 1) * dr;
      p.z1 = up ? zo + (p.rb - ro) / p.slope : zn + (p.rb - rn) / p.slope;
      p.i0 = up ? i_n - 1 : i_n + 1;
    } else {
      p.axi = true;
      const bool up = zo < k_n * dz;
      p.zb = (up ? k_n : k_n + 1) * dz;
      p.r2 = up ? ro + p.slope * (p.zb - zo) : rn + p.slope * (p.zb - zn);
      p.k0 = up ? k_n - 1 : k_n + 1;
    }
  } else if (res == 2) {
    // a path across a radial and an axial face; the other two-cell jumps are
    // too long for a step and are treated as the forward pass treats them
    const bool up = di > 0, right = dk > 0;
    if (di == 0 || (!up && dk == 0)) {
      p.ns = 0;
    } else {
      p.rad = p.axi = true;
      p.rb = (up ? i_n : i_n + 1) * dr;
      p.zb = (right ? k_n : k_n + 1) * dz;
      const bool from_new = !up && !right;
      p.z1 = from_new ? zn + (p.rb - rn) / p.slope : zo + (p.rb - ro) / p.slope;
      p.r2 = from_new ? rn + (p.zb - zn) * p.slope : ro + (p.zb - zo) * p.slope;
      p.ns = p.z1 == p.zb ? 0 : 3;
      p.rfirst = right ? p.z1 < p.zb : p.z1 > p.zb;
      p.i0 = up ? i_n - 1 : i_n + 1;
      p.k0 = right ? k_n - 1 : k_n + 1;
      p.i1 = p.rfirst ? i_n : p.i0;
      p.k1 = p.rfirst ? p.k0 : k_n;
    }
  } else if (res > 2) {
    p.ns = 0;
  }
  return p;
}

// reverse of the J_r / J_z deposit of the straight path (ro, zo) -> (rn, zn)
// (current_distribution, src/particles.cpp:480-685): the path is split at the
// radial face r = rb (met at z1) and the axial face z = zb (met at r2) that it
// crosses; with s the path parameter of the crossing, the adjoint of z1 goes
// to the ends as (1-s, s) along z and times -dz/dr along r, that of r2 likewise
__device__ __forceinline__ PieceAdj deposit_j_back(const GridDesc &g, const AdjGrid &lg, const StepScales &k, double q, double rn, double zn,
                                                   double ro, double zo) {
  const Path c = split_path(g, rn, zn, ro, zo);
  if (c.strict) {
    StrictSink sk{&g, &lg, {0.0, 0.0, 0.0, 0.0, 0.0}};
    strict_d(g, sk, cst(q), seed(rn, 0), seed(zn, 1), seed(ro, 2), seed(zo, 3));
    return sk.o;
  }
  const int ns = c.ns;
  const bool rfirst = c.rfirst;
  const double rb = c.rb, zb = c.zb, z1 = c.z1, r2 = c.r2, slope = c.slope;
  // the crossings in path order
  const double cr0 = rfirst ? rb : r2, cz0 = rfirst ? z1 : zb;
  const double cr1 = rfirst ? r2 : rb, cz1 = rfirst ? zb : z1;
  PieceAdj o{0.0, 0.0, 0.0, 0.0, 0.0};
  double c0r = 0.0, c0z = 0.0, c1r = 0.0, c1z = 0.0;  // adjoints of the crossings
#pragma nounroll
  for (int t = 0; t < ns; t++) {
    const bool first = t == 0, last = t == ns - 1;
    const PieceAdj p = segment_back(g, lg, k, last ? rn : first ? cr0 : cr1, last ? zn : first ? cz0 : cz1,
                                    first ? ro : t == 1 ? cr0 : cr1, first ? zo : t == 1 ? cz0 : cz1,
                                    last ? c.i_n : first ? c.i0 : c.i1, last ? c.k_n : first ? c.k0 : c.k1);
    o.s += p.s;
    if (first) {
      o.ro += p.ro;
      o.zo += p.zo;
    } else if (t == 1) {
      c0r += p.ro;
      c0z += p.zo;
    } else {
      c1r += p.ro;
      c1z += p.zo;
    }
    if (last) {
      o.rn += p.rn;
      o.zn += p.zn;
    } else if (first) {
      c0r += p.rn;
      c0z += p.zn;
    } else {
      c1r += p.rn;
      c1z += p.zn;
    }
  }
  if (c.rad) {
    const double l = rfirst ? c0z : c1z, s = (rb - ro) / (rn - ro), is = 1.0 / slope;
    o.zo += (1.0 - s) * l;
    o.zn += s * l;
    o.ro -= is * (1.0 - s) * l;
    o.rn -= is * s * l;
  }
  if (c.axi) {
    const double l = rfirst ? c1r : c0r, s = (zb - zo) / (zn - zo);
    o.ro += (1.0 - s) * l;
    o.rn += s * l;
    o.zo -= slope * (1.0 - s) * l;
    o.zn -= slope * s * l;
  }
  return o;
}

// reflection_single / Bunch::reflection_single on the half-step point; sx, sz:
// the signs that the reflections leave on (x, v_0) and (z, v_2)
__device__ __forceinline__ void walls_sign(const GridDesc &g, bool is_bunch, double &x, double &z, double &sx,
                                           double &sz, bool &alive) {
  const double dr = g.dr, dz = g.dz;
  const double radius_wall = g.r_size - dr / 2., longitude_wall = g.z_size - dz / 2.;
  sx = sz = 1.0;
  if (is_bunch) {
    if (x > radius_wall || z > longitude_wall) alive = false;
  } else {
    if (x > radius_wall) {
      x = radius_wall * 2. - x;
      sx = -sx;
    }
    if (z > longitude_wall) {
      z = longitude_wall * 2. - z;
      sz = -sz;
    }
  }
  if (x < dr / 2.) {
    x = dr - x;
    sx = -sx;
  }
  if (z < dz / 2.) {
    z = dz - z;
    sz = -sz;
  }
}

// the vector-Jacobian product of one living particle's step
template <bool VAY, class Box>
__device__ __forceinline__ void adj_particle(const GridDesc &g, const AdjFields &f, const AdjGrid &lg,
                                             const AdjSpecies &s, long long i, const AdjParticle &pt, const Box &box) {
  const double r0 = pt.r, z0 = pt.z, w = pt.w;
  const V3 v0 = {pt.vr, pt.vphi, pt.vz};
  const double half_dt = g.dt / 2.;
  const double es = s.k.es, bs = s.k.bs;
  V3 e, h;
  {
    const RingW wl = ring_lo(g, r0), wo = ring_own(g, r0);
    const ColW co = col_w(g, z0, false), ch = col_w(g, z0, true);
    e = es * V3{gather_grad(g, f.er, wl, co).v, gather_grad(g, f.ephi, wo, co).v, gather_grad(g, f.ez, wo, ch).v};
    h = bs * V3{gather_grad(g, f.hhr, wo, ch).v, gather_grad(g, f.hhphi, wl, ch).v, gather_grad(g, f.hhz, wl, co).v};
  }
  const V3 v = VAY ? vay_fwd(v0, e, h) : boris_fwd(v0, e, h);
  // first half step and rotation (step_v), then full_current_distribution
  const double x1 = r0 + v.x * half_dt, y = v.y * half_dt, z1 = z0 + v.z * half_dt;
  const double r1 = sqrt(x1 * x1 + y * y);
  double x2 = r1 + v.x * half_dt, z2 = z1 + v.z * half_dt, sx, sz;
  bool alive = true;
  walls_sign(g, Box::kBunch, x2, z2, sx, sz, alive);
  // adjoints: of v after the push, of the half-step point and of the start
  V3 lv = {0.0, 0.0, 0.0};
  double lr1 = 0.0, lz1 = 0.0, lr0 = 0.0, lz0 = 0.0, lw = 0.0;
  if (alive) {
    const double r2 = sqrt(x2 * x2 + y * y), ir2 = 1.0 / r2, st = y * ir2, ct = sqrt(1 - st * st);
    const double o0 = s.lvr[i], o1 = s.lvphi[i], o2 = s.lvz[i];
    const double vx = sx * v.x;  // after the walls
    // rotation of the velocity by the second half step's angle
    const double lst = vx * o1 - v.y * o0 - st / ct * (vx * o0 + v.y * o1);
    const PieceAdj p = deposit_j_back(g, lg, s.k, s.charge, r2, z2, r0, z0);
    lw += p.s;
    lr0 = w * p.ro;
    lz0 = w * p.zo;
    const double lr2 = s.lr[i] + w * p.rn - lst * st * ir2, lz2 = s.lz[i] + w * p.zn;
    const double lx2 = lr2 * x2 * ir2, ly2 = lr2 * st + lst * ir2;
    lr1 = sx * lx2;
    lz1 = sz * lz2;
    lv.x = sx * (ct * o0 + st * o1) + half_dt * lr1;
    lv.y = ct * o1 - st * o0 + half_dt * ly2;
    lv.z = sz * o2 + half_dt * lz1;
  }
  lw += jphi_back(g, lg.ljphi, s.k.kj, w, r1, z1, v.y, lr1, lz1, lv.y);
  const double ir1 = 1.0 / r1, lx1 = lr1 * x1 * ir1;
  lr0 += lx1;
  lz0 += lz1;
  lv.x += half_dt * lx1;
  lv.y += half_dt * (lr1 * y * ir1);
  lv.z += half_dt * lz1;
  V3 vb = v0, eb = e, hb = h;
  asm volatile("" : "+v"(vb.x), "+v"(vb.y), "+v"(vb.z), "+v"(eb.x), "+v"(eb.y), "+v"(eb.z), "+v"(hb.x), "+v"(hb.y), "+v"(hb.z));
  const PushBack p = VAY ? vay_back(vb, eb, hb, lv) : boris_back(vb, eb, hb, lv);
  const V3 le = es * p.e, lh = bs * p.b;
  double rg = r0, zg = z0;
  asm volatile("" : "+v"(rg), "+v"(zg));
  const RingW wl = ring_lo(g, rg), wo = ring_own(g, rg);
  const ColW co = col_w(g, zg, false), ch = col_w(g, zg, true);
  const Gathered e0 = gather_grad(g, f.er, wl, co), e1 = gather_grad(g, f.ephi, wo, co);
  const Gathered e2 = gather_grad(g, f.ez, wo, ch), h0 = gather_grad(g, f.hhr, wo, ch);
  const Gathered h1 = gather_grad(g, f.hhphi, wl, ch), h2 = gather_grad(g, f.hhz, wl, co);
  s.lr[i] = lr0 + (le.x * e0.dr + le.y * e1.dr + le.z * e2.dr + lh.x * h0.dr + lh.y * h1.dr + lh.z * h2.dr);
  s.lz[i] = lz0 + (le.x * e0.dz + le.y * e1.dz + le.z * e2.dz + lh.x * h0.dz + lh.y * h1.dz + lh.z * h2.dz);
  s.lvr[i] = p.v.x;
  s.lvphi[i] = p.v.y;
  s.lvz[i] = p.v.z;
  s.lw[i] += lw;
  box_scatter(g, box, 0, lg.ler, wl, co, le.x);
  box_scatter(g, box, 1, lg.lephi, wo, co, le.y);
  box_scatter(g, box, 2, lg.lez, wo, ch, le.z);
  box_scatter(g, box, 3, lg.lhr, wo, ch, lh.x);
  box_scatter(g, box, 4, lg.lhphi, wl, ch, lh.y);
  box_scatter(g, box, 5, lg.lhz, wl, co, lh.z);
}

#pragma clang fp contract(off)
template <bool VAY, bool BUNCH, bool F32>
__global__ void __launch_bounds__(256) k_adj_particles(GridDesc g, AdjFields f, AdjGrid lg, AdjSpecies s) {
  using Box = AdjBox<BUNCH>;
  constexpr int kSize = kABComp * Box::kR * kABK;
  __shared__ double box[kSize];
  const long long i = adj_slot<BUNCH>();
  AdjParticle pt;
  const bool live = i < s.n && adj_load<F32>(g, s.st, i, pt);
  int ci = INT_MAX, ck = INT_MAX;
  if (live) {
    ci = max(cell_r(g, pt.r), 0);
    ck = max(cell_z(g, pt.z), 0);
  }
  for (int t = threadIdx.x; t < kSize; t += blockDim.x) box[t] = 0.0;
  block_anchor<BUNCH, Box::kR, kABK>(ci, ck, live);
  const Box b{box, ci, ck};
  if (live) adj_particle<VAY>(g, f, lg, s, i, pt, b);
  else if (i < s.n) s.lr[i] = s.lz[i] = s.lvr[i] = s.lvphi[i] = s.lvz[i] = 0.0;
  __syncthreads();
  double *const lf[kABComp] = {lg.ler, lg.lephi, lg.lez, lg.lhr, lg.lhphi, lg.lhz};
  for (int t = threadIdx.x; t < kSize; t += blockDim.x) {
    const double v = box[t];
    if (v == 0.0) continue;
    const int comp = t / (Box::kR * kABK), rem = t - comp * Box::kR * kABK;
    const int gi = b.bi + rem / kABK, gk = b.bk + rem % kABK;
    // nodes off the grid never receive a stencil (the gathers clamp their cell)
    if ((unsigned)gi < (unsigned)g.nr && (unsigned)gk < (unsigned)g.nz)
      unsafeAtomicAdd(lf[comp] + (size_t)gi * (size_t)g.nz + gk, v);
  }
}

// ------------------------------------------------ tangent-linear (forward mode)
// The derivative of the same step along kDN tangent directions of the state,
// of the fields and of the weight: what does not depend on the direction (the
// push's intermediates, the gathers' and deposits' shares) is evaluated once,
// and each direction takes the linear maps between them, one direction after
// the other.  The tangents of the deposits (J-dot) are scattered with atomics.
// Together with the forward field updates applied to tangent grids this is the
// tangent-linear model of the loop, the exact transpose of what the adjoint
// above computes; <dphi/dw, dw> from the adjoint must equal the tangent of phi
// along dw to round-off (the dot-product test).  Re-executing the step in dual
// numbers of four directions took 256 + 66 registers, 736 bytes of scratch and a
// division per direction at every quotient: 184 us for 2.6e5 plasma particles
// and 55 us for 8e3 of a bunch; this form takes 63 and 33 us.
struct TlmFields {  // tangents of E^n and Hh^n, one set per direction
  const double *er[kDN], *ephi[kDN], *ez[kDN], *hhr[kDN], *hhphi[kDN], *hhz[kDN];
};
struct TlmJ {  // tangents of J^n, one set per direction
  double *jr[kDN], *jphi[kDN], *jz[kDN];
};
struct TlmSpecies {
  StateRef st;                          // state at step n (values)
  double *tr, *tz, *tvr, *tvphi, *tvz;  // kDN x n tangents: in at step n, out at n+1
  const double *tw;                     // kDN x n tangents of the weight
  double charge;
  StepScales k;
  long long n;                          // slots
};

// deposit tangents: every contribution v at node (i, k) adds its derivative
// part (one per direction) to the tangent J grids, through an LDS box of kR x
// kK nodes per component and direction (block_anchor; a particle's 48 global
// atomics, those of a bunch all on the same few nodes, were most of the kernel)
template <bool BUNCH>
struct TlmSink {
  static constexpr int kR = BUNCH ? 16 : 6, kK = BUNCH ? 32 : 64, kSize = 3 * kDN * kR * kK;
  const GridDesc *g;
  TlmJ j;
  double *box;  // LDS
  int bi, bk;   // node of box[.][0][0]
  // node (i, k): its place in a plane of the box, -1 outside the box, -2 off the grid
  __device__ __forceinline__ int node(int i, int k) const {
    if ((unsigned)i >= (unsigned)g->nr || (unsigned)k >= (unsigned)g->nz) return -2;
    const int li = i - bi, lk = k - bk;
    return (unsigned)li < (unsigned)kR && (unsigned)lk < (unsigned)kK ? li * kK + lk : -1;
  }
  __device__ __forceinline__ void put(int comp, int d, int node, int i, int k, double v) {
    if (node >= 0) {
      atomicAdd(box + (comp * kDN + d) * kR * kK + node, v);
    } else if (node == -1 && v != 0.0) {  // 0 along directions that do not reach the particle
      double *J = comp == kAR ? j.jr[d] : comp == kAPhi ? j.jphi[d] : j.jz[d];
      unsafeAtomicAdd(J + (size_t)i * (size_t)g->nz + (size_t)k, v);
    }
  }
  __device__ __forceinline__ void flush() const {
    for (int t = threadIdx.x; t < kSize; t += blockDim.x) {
      const double v = box[t];
      if (v == 0.0) continue;
      const int plane = t / (kR * kK), rem = t - plane * kR * kK;
      const int i = bi + rem / kK, k = bk + rem % kK, comp = plane / kDN, d = plane - comp * kDN;
      double *const *J = comp == kAR ? j.jr : comp == kAPhi ? j.jphi : j.jz;
      unsafeAtomicAdd(J[d] + (size_t)i * (size_t)g->nz + k, v);  // add() keeps off-grid nodes out
    }
  }
};

#pragma clang fp contract(fast)
// tangents of the push: the forward evaluation of boris_fwd / vay_fwd kept, and
// the map of one direction
struct BoostT {
  Boost b;
  bool x, y, z;  // components that are kept
};
__device__ __forceinline__ BoostT boost_t(V3 v) {
  return BoostT{boost_of(v), !(fabs(v.x) < kMnzl), !(fabs(v.y) < kMnzl), !(fabs(v.z) < kMnzl)};
}
__device__ __forceinline__ V3 along(const BoostT &t, V3 dv) {
  const V3 du = V3{t.x ? dv.x : 0.0, t.y ? dv.y : 0.0, t.z ? dv.z : 0.0};
  return fma3(per_c2(t.b.g0 * t.b.g0 * t.b.g0) * dot(t.b.u, du), t.b.u, t.b.g0 * du);
}
// tangent of inv_gamma(u) u, g = inv_gamma(u)
__device__ __forceinline__ V3 slow_t(double g, V3 u, V3 du) {
  return fma3(per_c2(-(g * g * g)) * dot(u, du), u, g * du);
}
struct BorisT {
  BoostT b0;
  V3 t, h, b, tp, w, u;
  double g1, c2, g2;
  __device__ __forceinline__ BorisT(V3 v, V3 e, V3 hs) : b0(boost_t(v)), h(hs) {
    t = fma3(b0.b.g0, b0.b.u, e);
    g1 = inv_gamma(t);
    b = g1 * h;
    tp = t + cross(t, b);
    c2 = 2.0 / (1.0 + dot(b, b));
    w = cross(tp, b);
    u = fma3(c2, w, t) + e;
    g2 = inv_gamma(u);
  }
  __device__ __forceinline__ V3 v() const { return g2 * u; }
  __device__ __forceinline__ V3 along_dir(V3 dv, V3 de, V3 dh) const {
    const V3 dt = along(b0, dv) + de;
    const V3 db = fma3(per_c2(-(g1 * g1 * g1)) * dot(t, dt), h, g1 * dh);
    const V3 dtp = dt + cross(dt, b) + cross(t, db);
    const V3 dw = cross(dtp, b) + cross(tp, db);
    const V3 du = fma3(-c2 * c2 * dot(b, db), w, fma3(c2, dw, dt + de));
    return slow_t(g2, u, du);
  }
};
struct VayT {
  BoostT b0;
  V3 t, h, th, up, b, q, u;
  double g1, ub, sg, root, al, s, al2, g3;
  __device__ __forceinline__ VayT(V3 v, V3 e, V3 hs) : b0(boost_t(v)), h(hs) {
    t = b0.b.g0 * b0.b.u;
    g1 = inv_gamma(t);
    th = cross(t, h);
    up = fma3(g1, th, t + e);
    const double B2 = dot(h, h);
    ub = dot(up, h);
    sg = 1.0 + per_c2(dot(up, up)) - B2;
    root = sqrt(sg * sg + 4. * (B2 + ub * ub));
    al = rsqrt_near(0.5 * (sg + root));
    b = al * h;
    s = 1.0 / (1.0 + dot(b, b));
    al2 = dot(up, b);
    q = fma3(al2, b, up) + cross(up, b);
    u = s * q;
    g3 = inv_gamma(u);
  }
  __device__ __forceinline__ V3 v() const { return g3 * u; }
  __device__ __forceinline__ V3 along_dir(V3 dv, V3 de, V3 dh) const {
    const V3 dt = along(b0, dv);
    const V3 dth = cross(dt, h) + cross(t, dh);
    const V3 dup = fma3(per_c2(-(g1 * g1 * g1)) * dot(t, dt), th, fma3(g1, dth, dt + de));
    const double dB2 = 2.0 * dot(h, dh), dub = dot(dup, h) + dot(up, dh);
    const double dsg = 2.0 / kC2 * dot(up, dup) - dB2;
    const double droot = (sg * dsg + 2.0 * dB2 + 4.0 * ub * dub) / root;
    const V3 db = fma3(-0.25 * al * al * al * (dsg + droot), h, al * dh);
    const double dal2 = dot(dup, b) + dot(up, db);
    const V3 dq = fma3(dal2, b, fma3(al2, db, dup)) + (cross(dup, b) + cross(up, db));
    return slow_t(g3, u, fma3(-2.0 * s * s * dot(b, db), q, s * dq));
  }
};

// tangents of the J_phi deposit (azimuthal_current_distribution,
// src/particles.cpp:688-784) of w charges q
template <class Sink>
__device__ __forceinline__ void jphi_tangent(const GridDesc &g, Sink &sk, double kj, double w, double r, double z,
                                             double vphi, const double (&tw)[kDN], const double (&tr)[kDN],
                                             const double (&tz)[kDN], const double (&tv)[kDN]) {
  const double dr = g.dr, dz = g.dz;
  const int i = max(cell_r(g, r), 0), k = max(cell_z(g, z), 0);
  const double r1 = r - 0.5 * dr, r2 = (i + 0.5) * dr, r3 = r + 0.5 * dr;
  const double i1 = (r > dr) ? vol_row(g, i).y : g.inv_cyl, i2 = vol_row(g, i + 1).y;
  const double d1 = (k + 0.5) * dz - (z - 0.5 * dz), d2 = (z + 0.5 * dz) - (k + 0.5) * dz;
  const double in = (r2 * r2 - r1 * r1) * i1, out = (r3 * r3 - r2 * r2) * i2;
  const double ir = 1.0 / r, K = kj * ir, P = w * K * vphi;
  const double din = P * (-2.0 * r1 * i1), dout = P * (2.0 * r3 * i2);
  const int n00 = sk.node(i, k), n10 = sk.node(i + 1, k), n01 = sk.node(i, k + 1), n11 = sk.node(i + 1, k + 1);
#pragma unroll
  for (int d = 0; d < kDN; d++) {
    const double c = K * (w * tv[d] + vphi * tw[d]) - P * ir * tr[d];
    const double ti = c * in + din * tr[d], to = c * out + dout * tr[d];
    const double zi = P * in * tz[d], zo = P * out * tz[d];
    sk.put(kAPhi, d, n00, i, k, ti * d1 - zi);
    sk.put(kAPhi, d, n10, i + 1, k, to * d1 - zo);
    sk.put(kAPhi, d, n01, i, k + 1, ti * d2 + zi);
    sk.put(kAPhi, d, n11, i + 1, k + 1, to * d2 + zo);
  }
}

// the tangents of a path's ends
struct PathT {
  double rn[kDN], zn[kDN], ro[kDN], zo[kDN], w[kDN];
};
// strict_d's sink in the tangent step (see StrictSink): w times the deposits of
// a unit weight, along each direction
template <class Sink>
struct StrictTangent {
  Sink *sk;
  const PathT *t;
  double w;
  __device__ __forceinline__ void add(int comp, int i, int k, D v) {
    const int n = sk->node(i, k);
#pragma unroll
    for (int d = 0; d < kDN; d++)
      sk->put(comp, d, n, i, k,
              w * (v.d[0] * t->rn[d] + v.d[1] * t->zn[d] + v.d[2] * t->ro[d] + v.d[3] * t->zo[d]) + v.v * t->w[d]);
  }
};

// tangents of the J_r / J_z deposit of w charges q on the path (ro, zo) -> (rn,
// zn), piece by piece (the closed forms above segment_back)
template <class Sink>
__device__ __forceinline__ void deposit_j_tangent(const GridDesc &g, Sink &sk, const StepScales &sc, double q, double w, double rn, double zn,
                                                  double ro, double zo, const PathT &t) {
  const double idr = g.inv_dr, idz = g.inv_dz;
  const Path c = split_path(g, rn, zn, ro, zo);
  if (c.strict) {
    const PathT own = t;  // t itself stays in registers
    StrictTangent<Sink> st{&sk, &own, w};
    strict_d(g, st, cst(q), seed(rn, 0), seed(zn, 1), seed(ro, 2), seed(zo, 3));
    return;
  }
  const double kz = sc.kz, kr = sc.kr;
  // path parameters of the crossings
  const double sr = c.rad ? (c.rb - ro) / (rn - ro) : 0.0, sz = c.axi ? (c.zb - zo) / (zn - zo) : 0.0;
  const double isl = c.rad ? 1.0 / c.slope : 0.0;
#pragma nounroll
  for (int n = 0; n < c.ns; n++) {
    const bool first = n == 0, last = n == c.ns - 1;
    // the piece ends at crossing n and begins at crossing n - 1; crossing n is
    // the radial face's if
    const bool nrad = first == c.rfirst, orad = (n == 1) == c.rfirst;
    const double prn = last ? rn : nrad ? c.rb : c.r2, pzn = last ? zn : nrad ? c.z1 : c.zb;
    const double pro = first ? ro : orad ? c.rb : c.r2, pzo = first ? zo : orad ? c.z1 : c.zb;
    const int i = last ? c.i_n : first ? c.i0 : c.i1, k = last ? c.k_n : first ? c.k0 : c.k1;
    if ((fabs(prn - pro) < kMnzl) || (fabs(pzn - pzo) < kMnzl)) continue;
    const double fi = (double)i;
    const double a = per_dr(g, pro) - fi, b = per_dz(g, pzo) - (double)k;
    const double drho = per_dr(g, prn - pro), dzeta = per_dz(g, pzn - pzo);
    const double hdr = 0.5 * drho, ub = 1.0 - b, qdz = 0.25 * dzeta, p0 = 0.5 * ub - qdz, p1 = 0.5 * b + qdz;
    // J_z = kz w dzeta (z0, z1), J_r = kr w (j0, j1); along a direction, with
    // the tangents (ta, tb, tdr, tdz) of (a, b, drho, dzeta):
    //   z0' = z0a ta + z0d tdr, j0' = j0a ta + j0b tb + j0d tdr + j0z tdz, and so on
    double z0, z1, j0, j1, z0a, z1a, z0d, z1d, j0a, j1a, jb, j0d, j1d, jz;
    if (i == 0) {
      z0 = 8.0 * (1.0 - hdr - a);
      z1 = hdr + 1.0 + a;
      z0a = -8.0;
      z1a = 1.0;
      z0d = -4.0;
      z1d = 0.5;
      j0 = 2.0 * drho * p0;
      j1 = 2.0 * drho * p1;
      j0a = j1a = 0.0;
      jb = drho;
      j0d = 2.0 * p0;
      j1d = 2.0 * p1;
      jz = hdr;
    } else {
      const double i0 = 1.0 / fi, i1 = 1.0 / (fi + 1.0), ih = 1.0 / (fi + 0.5);
      const double rs = fi + a, re = rs + drho, irs = 1.0 / rs, ire = 1.0 / re;
      const double ii = fi * (fi + 1.0), x = drho * irs, u = drho * ire;
      double M, dM;
      m_and_slope(x, M, dM);
      const double N = -u - M, iiM = ii * M, cc = 0.5 * ii * irs;
      const double A0 = (1.0 - a) * (2.0 * fi + a) + iiM, A1 = a * (2.0 * fi + 1.0 + a) - iiM;
      const double R0 = u * ub + dzeta * N, R1 = u * b - dzeta * N;
      // derivatives of x, u and N along a and drho
      const double xa = -x * irs, ua = -u * ire, ud = rs * ire * ire, Ma = dM * xa, Md = dM * irs;
      const double Na = -ua - Ma, Nd = -ud - Md;
      z0 = (A0 * irs - hdr) * i0;
      z1 = (A1 * irs + hdr) * i1;
      z0a = (((1.0 - 2.0 * fi - 2.0 * a) + ii * Ma) - A0 * irs) * irs * i0;
      z1a = (((2.0 * fi + 1.0 + 2.0 * a) - ii * Ma) - A1 * irs) * irs * i1;
      z0d = (ii * Md * irs - 0.5) * i0;
      z1d = (0.5 - ii * Md * irs) * i1;
      j0 = (drho * p0 + cc * R0) * ih;
      j1 = (drho * p1 + cc * R1) * ih;
      j0a = cc * (ua * ub + dzeta * Na - R0 * irs) * ih;
      j1a = cc * (ua * b - dzeta * Na - R1 * irs) * ih;
      jb = (hdr + cc * u) * ih;
      j0d = (p0 + cc * (ud * ub + dzeta * Nd)) * ih;
      j1d = (p1 + cc * (ud * b - dzeta * Nd)) * ih;
      jz = (0.25 * drho - cc * N) * ih;
    }
    const int n00 = sk.node(i, k), n10 = sk.node(i + 1, k), n01 = sk.node(i, k + 1);
    const double wz = w * kz, wr = w * kr;
#pragma unroll
    for (int d = 0; d < kDN; d++) {
      double ern = t.rn[d], ezn = t.zn[d], ero = t.ro[d], ezo = t.zo[d];
      if (c.ns > 1) {
        // with s the path parameter of a crossing, the one with the radial
        // face moves along z, that with the axial face along r
        const double tz1 = (1.0 - sr) * ezo + sr * ezn - isl * ((1.0 - sr) * ero + sr * ern);
        const double tr2 = (1.0 - sz) * ero + sz * ern - c.slope * ((1.0 - sz) * ezo + sz * ezn);
        if (!last) {
          ern = nrad ? 0.0 : tr2;
          ezn = nrad ? tz1 : 0.0;
        }
        if (!first) {
          ero = orad ? 0.0 : tr2;
          ezo = orad ? tz1 : 0.0;
        }
      }
      const double ta = ero * idr, tb = ezo * idz, tdr = (ern - ero) * idr, tdz = (ezn - ezo) * idz;
      const double f = wz * tdz + kz * t.w[d] * dzeta, e = wz * dzeta, h = kr * t.w[d];
      const double m = jb * tb + jz * tdz;
      sk.put(kAZ, d, n00, i, k, f * z0 + e * (z0a * ta + z0d * tdr));
      sk.put(kAZ, d, n10, i + 1, k, f * z1 + e * (z1a * ta + z1d * tdr));
      sk.put(kAR, d, n00, i, k, h * j0 + wr * (j0a * ta + j0d * tdr - m));
      sk.put(kAR, d, n01, i, k + 1, h * j1 + wr * (j1a * ta + j1d * tdr + m));
    }
  }
}

template <class Push, bool BUNCH, class Sink>
__device__ __forceinline__ void tlm_particle(const GridDesc &g, const AdjFields &f, const TlmFields &tf, Sink &sk,
                                             const TlmSpecies &s, long long i, const AdjParticle &pt) {
  const long long n = s.n;
  const double r0 = pt.r, z0 = pt.z, w = pt.w, half_dt = g.dt / 2.;
  const double es = s.k.es, bs = s.k.bs;
  const RingW wl = ring_lo(g, r0), wo = ring_own(g, r0);
  const ColW co = col_w(g, z0, false), ch = col_w(g, z0, true);
  const Gathered e0 = gather_grad(g, f.er, wl, co), e1 = gather_grad(g, f.ephi, wo, co);
  const Gathered e2 = gather_grad(g, f.ez, wo, ch), h0 = gather_grad(g, f.hhr, wo, ch);
  const Gathered h1 = gather_grad(g, f.hhphi, wl, ch), h2 = gather_grad(g, f.hhz, wl, co);
  const Push push(V3{pt.vr, pt.vphi, pt.vz}, es * V3{e0.v, e1.v, e2.v}, bs * V3{h0.v, h1.v, h2.v});
  const V3 v = push.v();
  // first half step and rotation (step_v), then full_current_distribution
  const double x1 = r0 + v.x * half_dt, y = v.y * half_dt, z1 = z0 + v.z * half_dt;
  const double r1 = sqrt(x1 * x1 + y * y), ir1 = 1.0 / r1;
  double x2 = r1 + v.x * half_dt, z2 = z1 + v.z * half_dt, sx, sz;
  bool alive = true;
  walls_sign(g, BUNCH, x2, z2, sx, sz, alive);
  const double r2 = sqrt(x2 * x2 + y * y), ir2 = 1.0 / r2, st = y * ir2, ct = sqrt(1 - st * st);
  const double vx = sx * v.x;  // after the walls
  PathT t;
  double tr1[kDN], tz1[kDN], tvp[kDN];  // at the J_phi deposit
#pragma unroll
  for (int d = 0; d < kDN; d++) {
    const size_t p = (size_t)d * n + i;
    const double tr = s.tr[p], tz = s.tz[p];
    t.ro[d] = tr;
    t.zo[d] = tz;
    t.w[d] = s.tw[p];
    const V3 de = es * V3{tr * e0.dr + tz * e0.dz + gather_grad(g, tf.er[d], wl, co).v,
                          tr * e1.dr + tz * e1.dz + gather_grad(g, tf.ephi[d], wo, co).v,
                          tr * e2.dr + tz * e2.dz + gather_grad(g, tf.ez[d], wo, ch).v};
    const V3 dh = bs * V3{tr * h0.dr + tz * h0.dz + gather_grad(g, tf.hhr[d], wo, ch).v,
                          tr * h1.dr + tz * h1.dz + gather_grad(g, tf.hhphi[d], wl, ch).v,
                          tr * h2.dr + tz * h2.dz + gather_grad(g, tf.hhz[d], wl, co).v};
    const V3 dv = push.along_dir(V3{s.tvr[p], s.tvphi[p], s.tvz[p]}, de, dh);
    const double ty = dv.y * half_dt;
    tr1[d] = (x1 * (tr + dv.x * half_dt) + y * ty) * ir1;
    tz1[d] = tz + dv.z * half_dt;
    tvp[d] = dv.y;
    const double tx2 = sx * (tr1[d] + dv.x * half_dt);
    t.rn[d] = (x2 * tx2 + y * ty) * ir2;
    t.zn[d] = sz * (tz1[d] + dv.z * half_dt);
    // rotation of the velocity by the second half step's angle
    const double ts = (ty - st * t.rn[d]) * ir2, tc = -st / ct * ts, tvx = sx * dv.x;
    s.tr[p] = alive ? t.rn[d] : 0.0;
    s.tz[p] = alive ? t.zn[d] : 0.0;
    s.tvr[p] = alive ? tc * vx + ct * tvx - ts * v.y - st * dv.y : 0.0;
    s.tvphi[p] = alive ? ts * vx + st * tvx + tc * v.y + ct * dv.y : 0.0;
    s.tvz[p] = alive ? sz * dv.z : 0.0;
    __builtin_amdgcn_sched_barrier(0);  // one direction's registers at a time
  }
  jphi_tangent(g, sk, s.k.kj, w, r1, z1, v.y, t.w, tr1, tz1, tvp);
  if (alive) deposit_j_tangent(g, sk, s.k, s.charge, w, r2, z2, r0, z0, t);
}
#pragma clang fp contract(off)

template <bool VAY, bool BUNCH, bool F32>
__global__ void __launch_bounds__(256) k_tlm_particles(GridDesc g, AdjFields f, TlmFields tf, TlmJ tj, TlmSpecies s) {
  using Sink = TlmSink<BUNCH>;
  __shared__ double box[Sink::kSize];
  const long long i = adj_slot<BUNCH>();
  AdjParticle pt;
  const bool live = i < s.n && adj_load<F32>(g, s.st, i, pt);
  int ci = INT_MAX, ck = INT_MAX;
  if (live) {
    ci = max(cell_r(g, pt.r), 0);
    ck = max(cell_z(g, pt.z), 0);
  }
  for (int t = threadIdx.x; t < Sink::kSize; t += blockDim.x) box[t] = 0.0;
  block_anchor<BUNCH, Sink::kR, Sink::kK>(ci, ck, live);
  Sink sk{&g, tj, box, ci, ck};
  if (live) {
    tlm_particle<typename std::conditional<VAY, VayT, BorisT>::type, BUNCH>(g, f, tf, sk, s, i, pt);
  } else if (i < s.n) {
    // dead (or padding) slots keep zero tangents; a particle injected later
    // starts with zero tangents, as its injected state does not depend on w
#pragma unroll
    for (int d = 0; d < kDN; d++) {
      const size_t p = (size_t)d * s.n + i;
      s.tr[p] = s.tz[p] = s.tvr[p] = s.tvphi[p] = s.tvz[p] = 0.0;
    }
  }
  __syncthreads();
  sk.flush();
}

// tangent of the objective: phi_dot[d] += scale * sum 2 E_z(0, k) E_z-dot_d(0, k)
// over k0..k1, and phi += scale * sum E_z(0,k)^2 (one block)
__global__ void __launch_bounds__(256) k_tlm_objective(GridDesc g, const double *ez, const double *ezd0,
                                                       const double *ezd1, const double *ezd2, const double *ezd3,
                                                       int k0, int k1, double scale, double *phi) {
  __shared__ double part[5][256];
  double acc[5] = {0, 0, 0, 0, 0};
  const double *ezd[4] = {ezd0, ezd1, ezd2, ezd3};
  for (int k = k0 + threadIdx.x; k <= k1; k += blockDim.x) {
    const double e = ez[k];
    acc[0] += scale * e * e;
#pragma unroll
    for (int d = 0; d < 4; d++) acc[1 + d] += scale * 2.0 * e * ezd[d][k];
  }
#pragma unroll
  for (int a = 0; a < 5; a++) part[a][threadIdx.x] = acc[a];
  __syncthreads();
  for (int s2 = 128; s2 > 0; s2 >>= 1) {
    if ((int)threadIdx.x < s2)
#pragma unroll
      for (int a = 0; a < 5; a++) part[a][threadIdx.x] += part[a][threadIdx.x + s2];
    __syncthreads();
  }
  if (threadIdx.x < 5) phi[threadIdx.x] += part[threadIdx.x][0];
}

// ------------------------------------------------------------- the fields

struct AdjE {  // adjoints of E, H (after step), Hh, J and the coefficients; E of the pass before: ler.., scaled: ser..
  double *ler, *lephi, *lez, *lhr, *lhphi, *lhz, *lhhr, *lhhphi, *lhhz, *ljr, *ljphi, *ljz;
  double *ser, *sephi, *sez;
  const double *ke, *kh;
};

__device__ __forceinline__ size_t at(const GridDesc &g, int i, int k) { return (size_t)i * (size_t)g.nz + (size_t)k; }

// which E entries EField::calc_field updates (src/eField.cpp:99-168)
__device__ __forceinline__ bool upd_er(const GridDesc &g, int i, int k) { return i <= g.nr - 2 && k >= 1 && k <= g.nz - 2; }
__device__ __forceinline__ bool upd_ephi(const GridDesc &g, int i, int k) {
  return i >= 1 && i <= g.nr - 2 && k >= 1 && k <= g.nz - 2;
}
__device__ __forceinline__ bool upd_ez(const GridDesc &g, int i, int k) { return i <= g.nr - 2 && k <= g.nz - 2; }

// step 1, with step 3b of the iteration after it (lambda_H <- lambda_H +
// lambda_Hh, lambda_Hh <- 0, each node its own): lambda_H += C^T (Kh lambda_E),
// lambda_J = -Kh lambda_E (pull form: each H node sums the E nodes whose update
// reads it), and lambda_E scaled by Ke on the updated entries into the other
// set of E grids, as the neighbours still read this one
__global__ void __launch_bounds__(256) k_adj_e_curl(GridDesc g, AdjE a) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y;
  if (k >= g.nz) return;
  const double dr = g.dr, dz = g.dz;
  const size_t p = at(g, i, k);
  // J adjoints
  a.ljr[p] = upd_er(g, i, k) ? -a.kh[p] * a.ler[p] : 0.0;
  a.ljphi[p] = upd_ephi(g, i, k) ? -a.kh[p] * a.lephi[p] : 0.0;
  a.ljz[p] = upd_ez(g, i, k) ? -a.kh[p] * a.lez[p] : 0.0;
  // H_phi(i, k): E_r(i, k) has -Kh (H_phi(i,k) - H_phi(i,k-1)) / dz, E_r(i, k+1)
  // the same with k+1; E_z(i, k) has +Kh ((H_phi(i,k) - H_phi(i-1,k)) / dr +
  // (H_phi(i,k) + H_phi(i-1,k)) / (2 dr i)) for i >= 1 and +Kh 4/dr H_phi(0,k)
  // on the axis; E_z(i+1, k) the same with i+1
  double lhphi = 0.0;
  if (upd_er(g, i, k)) lhphi += -a.kh[p] / dz * a.ler[p];
  if (k + 1 < g.nz && upd_er(g, i, k + 1)) lhphi += a.kh[p + 1] / dz * a.ler[p + 1];
  if (upd_ez(g, i, k)) {
    if (i == 0)
      lhphi += a.kh[p] * (4.0 / dr) * a.lez[p];
    else
      lhphi += a.kh[p] * (1.0 / dr + 1.0 / (2.0 * dr * i)) * a.lez[p];
  }
  if (i + 1 < g.nr && upd_ez(g, i + 1, k)) {
    const size_t pu = p + g.nz;
    lhphi += a.kh[pu] * (-1.0 / dr + 1.0 / (2.0 * dr * (i + 1))) * a.lez[pu];
  }
  a.lhphi[p] = (a.lhphi[p] + a.lhhphi[p]) + lhphi;
  // H_r(i, k): E_phi(i, k) has +Kh (H_r(i,k) - H_r(i,k-1)) / dz, E_phi(i, k+1) -
  double lhr = 0.0;
  if (upd_ephi(g, i, k)) lhr += a.kh[p] / dz * a.lephi[p];
  if (k + 1 < g.nz && upd_ephi(g, i, k + 1)) lhr += -a.kh[p + 1] / dz * a.lephi[p + 1];
  a.lhr[p] = (a.lhr[p] + a.lhhr[p]) + lhr;
  // H_z(i, k): E_phi(i, k) has -Kh (H_z(i,k) - H_z(i-1,k)) / dr, E_phi(i+1, k) +
  double lhz = 0.0;
  if (upd_ephi(g, i, k)) lhz += -a.kh[p] / dr * a.lephi[p];
  if (i + 1 < g.nr && upd_ephi(g, i + 1, k)) lhz += a.kh[p + g.nz] / dr * a.lephi[p + g.nz];
  a.lhz[p] = (a.lhz[p] + a.lhhz[p]) + lhz;
  a.lhhr[p] = 0.0;
  a.lhhphi[p] = 0.0;
  a.lhhz[p] = 0.0;
  a.ser[p] = upd_er(g, i, k) ? a.ler[p] * a.ke[p] : a.ler[p];
  a.sephi[p] = upd_ephi(g, i, k) ? a.lephi[p] * a.ke[p] : a.lephi[p];
  a.sez[p] = upd_ez(g, i, k) ? a.lez[p] * a.ke[p] : a.lez[p];
}

// step 3a: lambda_alpha = lambda_H + lambda_Hh / 2 (H_z: -(...)), pulled into
// lambda_E through A^T (HField::calc_field, src/hField.cpp:93-157):
//   H_r(i,k),   i <= nr-1, k <= nz-2: alpha = dt (E_phi(i,k+1) - E_phi(i,k)) / (dz mu0)
//   H_phi(i,k), i <= nr-2, k <= nz-2: alpha = dt ((E_z(i+1,k) - E_z(i,k)) / dr - (E_r(i,k+1) - E_r(i,k)) / dz) / mu0
//   H_z(i,k),   i <= nr-2, k <= nz-2: H_z -= alpha, alpha = dt ((E_phi(i+1,k) + E_phi(i,k)) / (2 dr (i+1/2))
//                                                   + (E_phi(i+1,k) - E_phi(i,k)) / dr) / mu0
__global__ void __launch_bounds__(256) k_adj_h(GridDesc g, AdjE a) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y;
  if (k >= g.nz) return;
  const double dt = g.dt, dr = g.dr, dz = g.dz, mu = kMagnConst;
  const size_t p = at(g, i, k);
  auto la_r = [&](int ii, int kk) {  // lambda_alpha of H_r at (ii, kk), 0 outside its update domain
    if (ii < 0 || ii > g.nr - 1 || kk < 0 || kk > g.nz - 2) return 0.0;
    const size_t q = at(g, ii, kk);
    return a.lhr[q] + 0.5 * a.lhhr[q];
  };
  auto la_phi = [&](int ii, int kk) {
    if (ii < 0 || ii > g.nr - 2 || kk < 0 || kk > g.nz - 2) return 0.0;
    const size_t q = at(g, ii, kk);
    return a.lhphi[q] + 0.5 * a.lhhphi[q];
  };
  auto la_z = [&](int ii, int kk) {
    if (ii < 0 || ii > g.nr - 2 || kk < 0 || kk > g.nz - 2) return 0.0;
    const size_t q = at(g, ii, kk);
    return -(a.lhz[q] + 0.5 * a.lhhz[q]);
  };
  // E_phi(i,k): H_r(i,k-1) +dt/(dz mu), H_r(i,k) -dt/(dz mu);
  // H_z(i-1,k): dt/mu (1/(2 dr (i-1/2)) + 1/dr); H_z(i,k): dt/mu (1/(2 dr (i+1/2)) - 1/dr)
  double le_phi = dt / (dz * mu) * (la_r(i, k - 1) - la_r(i, k));
  if (i >= 1) le_phi += dt / mu * (1.0 / (2.0 * dr * (i - 0.5)) + 1.0 / dr) * la_z(i - 1, k);
  le_phi += dt / mu * (1.0 / (2.0 * dr * (i + 0.5)) - 1.0 / dr) * la_z(i, k);
  // E_z(i,k): H_phi(i-1,k) +dt/(dr mu), H_phi(i,k) -dt/(dr mu)
  double le_z = dt / (dr * mu) * (la_phi(i - 1, k) - la_phi(i, k));
  // E_r(i,k): H_phi(i,k-1) -dt/(dz mu), H_phi(i,k) +dt/(dz mu)
  double le_r = dt / (dz * mu) * (la_phi(i, k) - la_phi(i, k - 1));
  a.ser[p] += le_r;
  a.sephi[p] += le_phi;
  a.sez[p] += le_z;
}

// objective seed: lambda_Ez(0, k) += scale * 2 E_z(0, k) on k0..k1, and the
// objective's sum scale * sum E_z(0,k)^2 into *phi (one block)
__global__ void __launch_bounds__(256) k_adj_seed(GridDesc g, const double *ez, double *lez, int k0, int k1, double scale,
                                                  double *phi) {
  __shared__ double part[256];
  double acc = 0.0;
  for (int k = k0 + threadIdx.x; k <= k1; k += blockDim.x) {
    const double e = ez[k];  // row 0
    lez[k] += scale * 2.0 * e;
    acc += scale * e * e;
  }
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *phi += part[0];
}

// several device-to-device copies in one launch (grid.y: the copy), 16 bytes a
// thread and pass
constexpr int kCopies = 24;
struct CopyArgs {
  CopySeg seg[kCopies];
};
__global__ void __launch_bounds__(256) k_copy(CopyArgs a) {
  const CopySeg s = a.seg[blockIdx.y];
  const size_t n = s.bytes / sizeof(uint4), stride = (size_t)gridDim.x * blockDim.x;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t i = t; i < n; i += stride) ((uint4 *)s.dst)[i] = ((const uint4 *)s.src)[i];
  if (t < s.bytes - n * sizeof(uint4)) ((uint8_t *)s.dst)[n * sizeof(uint4) + t] = ((const uint8_t *)s.src)[n * sizeof(uint4) + t];
}

}  // namespace

// ------------------------------------------------------------- launchers

void launch_copies(const std::vector<CopySeg> &segs, hipStream_t st) {
  for (size_t at = 0; at < segs.size(); at += kCopies) {
    CopyArgs a;
    const int n = (int)std::min<size_t>(kCopies, segs.size() - at);
    size_t most = 0;
    for (int j = 0; j < n; j++) {
      a.seg[j] = segs[at + j];
      most = std::max(most, a.seg[j].bytes);
    }
    const unsigned blocks = (unsigned)std::min<size_t>(1024, most / (sizeof(uint4) * 256) + 1);
    hipLaunchKernelGGL(k_copy, dim3(blocks, n), dim3(256), 0, st, a);
  }
}

AdjE adj_e(double *const *lam, double *const *scaled, const double *ke, const double *kh) {
  return AdjE{lam[0], lam[1], lam[2], lam[3], lam[4], lam[5], lam[6], lam[7], lam[8], lam[9], lam[10], lam[11],
              scaled[0], scaled[1], scaled[2], ke, kh};
}

void launch_adj_fields_pre(const GridDesc &g, double *const *lam, double *const *scaled, const double *ke,
                           const double *kh, hipStream_t st) {
  dim3 grid((g.nz + 255) / 256, g.nr);
  hipLaunchKernelGGL(k_adj_e_curl, grid, dim3(256), 0, st, g, adj_e(lam, scaled, ke, kh));
}

void launch_adj_fields_post(const GridDesc &g, double *const *lam, double *const *scaled, const double *ke,
                            const double *kh, hipStream_t st) {
  dim3 grid((g.nz + 255) / 256, g.nr);
  hipLaunchKernelGGL(k_adj_h, grid, dim3(256), 0, st, g, adj_e(lam, scaled, ke, kh));
}

void launch_adj_particles(const GridDesc &g, const double *const *fields6, double *const *lam, double *const *scaled,
                          const StateRef &state, double *const *lstate, double *lw, double charge, double mass,
                          long long n, int is_bunch, int pusher, hipStream_t st) {
  if (n <= 0) return;
  AdjFields f{fields6[0], fields6[1], fields6[2], fields6[3], fields6[4], fields6[5]};
  AdjGrid lg{lam[9], lam[10], lam[11], scaled[0], scaled[1], scaled[2], lam[6], lam[7], lam[8]};
  AdjSpecies s{state, lstate[0], lstate[1], lstate[2], lstate[3], lstate[4], lw, charge, scales_of(g, charge, mass, pusher == 1), n};
  const dim3 grid((unsigned)((n + 255) / 256));
  using K = void (*)(GridDesc, AdjFields, AdjGrid, AdjSpecies);
  static const K kernels[8] = {k_adj_particles<false, false, false>, k_adj_particles<true, false, false>,
                               k_adj_particles<false, true, false>,  k_adj_particles<true, true, false>,
                               k_adj_particles<false, false, true>,  k_adj_particles<true, false, true>,
                               k_adj_particles<false, true, true>,   k_adj_particles<true, true, true>};
  hipLaunchKernelGGL(kernels[(pusher == 1) + 2 * (is_bunch != 0) + 4 * state.f32], grid, dim3(256), 0, st,
                     g, f, lg, s);
}

void launch_adj_seed(const GridDesc &g, const double *ez, double *lez, int k0, int k1, double scale, double *phi,
                     hipStream_t st) {
  hipLaunchKernelGGL(k_adj_seed, dim3(1), dim3(256), 0, st, g, ez, lez, k0, k1, scale, phi);
}

void launch_tlm_particles(const GridDesc &g, const double *const *fields6, double *const *const *tgrid,
                          const StateRef &state, double *const *tstate, const double *tw, double charge, double mass,
                          long long n, int is_bunch, int pusher, hipStream_t st) {
  if (n <= 0) return;
  AdjFields f{fields6[0], fields6[1], fields6[2], fields6[3], fields6[4], fields6[5]};
  TlmFields tf;
  TlmJ tj;
  for (int d = 0; d < kDN; d++) {
    double *const *a = tgrid[d];
    tf.er[d] = a[kER];
    tf.ephi[d] = a[kEPhi];
    tf.ez[d] = a[kEZ];
    tf.hhr[d] = a[kHHR];
    tf.hhphi[d] = a[kHHPhi];
    tf.hhz[d] = a[kHHZ];
    tj.jr[d] = a[kJR];
    tj.jphi[d] = a[kJPhi];
    tj.jz[d] = a[kJZ];
  }
  TlmSpecies s{state, tstate[0], tstate[1], tstate[2], tstate[3], tstate[4], tw, charge, scales_of(g, charge, mass, pusher == 1), n};
  const dim3 grid((unsigned)((n + 255) / 256));
  using K = void (*)(GridDesc, AdjFields, TlmFields, TlmJ, TlmSpecies);
  static const K kernels[8] = {k_tlm_particles<false, false, false>, k_tlm_particles<true, false, false>,
                               k_tlm_particles<false, true, false>,  k_tlm_particles<true, true, false>,
                               k_tlm_particles<false, false, true>,  k_tlm_particles<true, false, true>,
                               k_tlm_particles<false, true, true>,   k_tlm_particles<true, true, true>};
  const int k = (pusher == 1) + 2 * (is_bunch != 0) + 4 * state.f32;
  hipLaunchKernelGGL(kernels[k], grid, dim3(256), 0, st, g, f, tf, tj, s);
}

void launch_tlm_objective(const GridDesc &g, const double *ez, double *const *const *tgrid, int k0, int k1,
                          double scale, double *phi5, hipStream_t st) {
  hipLaunchKernelGGL(k_tlm_objective, dim3(1), dim3(256), 0, st, g, ez, tgrid[0][kEZ], tgrid[1][kEZ],
                     tgrid[2][kEZ], tgrid[3][kEZ], k0, k1, scale, phi5);
}

}  // namespace pdp3
