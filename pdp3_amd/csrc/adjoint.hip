// Hand-written adjoint of one loop iteration (src/loadInitParam.cpp:471-587)
// in the FP64 plain form's arithmetic, for gradients of a field objective with
// respect to the particle weights.
//
// Forward iteration n:  H^{n+1} = H^n + A E^n, Hh^n = H^n + A E^n / 2
//                       (x, v)^{n+1}, J^n = P((x, v)^n, E^n, Hh^n, w)
//                       E^{n+1} = Ke E^n - Kh (J^n - C H^{n+1})
// Backward, given the adjoints of E^{n+1}, H^{n+1} and the particle states:
//   1. lambda_J = -Kh lambda_E;  lambda_H += C^T (Kh lambda_E);  lambda_E <- Ke lambda_E
//   2. per particle, the vector-Jacobian product of P: the particle's step is
//      re-executed in dual numbers (value + N directional derivatives) over
//      its 12 inputs (r, z, v, the gathered E and H, w) in 12/N passes; every
//      output (new r, z, v and each grid deposit) contributes its adjoint
//      times its derivative; the adjoints of the gathered fields are scattered
//      back to the nodes with the gather weights, the weight adjoint is
//      accumulated per particle
//   3. lambda_alpha = lambda_H + lambda_Hh / 2;  lambda_E += A^T lambda_alpha;
//      lambda_H <- lambda_H + lambda_Hh
// The operators A (HField::calc_field, src/hField.cpp:93-157), C, Ke, Kh
// (EField::calc_field, src/eField.cpp:85-170, PML in Ke / Kh) are transposed
// node by node in pull form (no atomics).  The particle step follows
// particles_fp64.hip expression for expression.
#include <algorithm>
#include <climits>

#include "context.hpp"
#include "crmath.hpp"
#include "sink.hpp"

namespace pdp3 {

namespace {

constexpr int kDN = 4;  // directions
static_assert(kDN == kTangentDirs, "the tangent-linear model runs one direction per dual slot");

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
__device__ __forceinline__ D dsqrt(D a) {
  D r;
  r.v = sqrt(a.v);
  const double h = 0.5 / r.v;
  for (int j = 0; j < kDN; j++) r.d[j] = a.d[j] * h;
  return r;
}
__device__ __forceinline__ D dlog(D a) {
  D r;
  r.v = log(a.v);
  for (int j = 0; j < kDN; j++) r.d[j] = a.d[j] / a.v;
  return r;
}
// pow(y, -0.5) of lib::get_gamma_inv with the correctly rounded value
__device__ __forceinline__ D drsqrt(D a) {
  D r;
  r.v = rsqrt_cr(a.v);
  const double h = -0.5 * r.v * r.v * r.v;
  for (int j = 0; j < kDN; j++) r.d[j] = a.d[j] * h;
  return r;
}

constexpr double kC2 = kLightSpeed * kLightSpeed;

// ------------------------------------------------------------ the particle

struct AdjFields {
  const double *er, *ephi, *ez, *hhr, *hhphi, *hhz;  // E^n, Hh^n
};
struct AdjGrid {
  const double *ljr, *ljphi, *ljz;             // adjoint of J^n
  double *ler, *lephi, *lez, *lhr, *lhphi, *lhz;  // adjoint of E^n, Hh^n (scatter, atomics)
};
struct AdjSpecies {
  StateRef st;                          // state at step n
  double *lr, *lz, *lvr, *lvphi, *lvz;  // in: adjoint of the state after step n; out: before
  double *lw;                           // accumulated adjoint of the weight
  double charge, mass;
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

__device__ __forceinline__ int cell_number(double x, double dx) { return (int)ceil(x / dx) - 1; }
__device__ __forceinline__ double cell_volume(int i, double dr, double dz) { return kPi * dz * dr * dr * 2.0 * i; }
__device__ __forceinline__ double cyl_vol(double z, double r) { return kPi * z * r * r / 4.; }

// the node weights of the four-node gather (src/eField.cpp:204-316) for one
// component family; weights[] multiply F at (i_r, k), (i_r+1, k), (i_r, k+1),
// (i_r+1, k+1).  Dual in (r, z).
struct GatherW {
  int ir, kz;
  D w[4];
};
__device__ GatherW gather_w(const GridDesc &g, D radius, D longitude, bool lo, bool zhalf) {
  const double dr = g.dr, dz = g.dz;
  D r1 = radius - 0.5 * dr;
  D r3 = radius + 0.5 * dr;
  int i_r = lo ? cell_number(radius.v - 0.5 * dr, dr) : cell_number(radius.v, dr);
  int k_z = zhalf ? cell_number(longitude.v - 0.5 * dz, dz) : cell_number(longitude.v, dz);
  if (i_r < 0) i_r = 0;
  if (k_z < 0) k_z = 0;
  i_r = min(i_r, g.nr - 2);
  k_z = min(k_z, g.nz - 2);
  double vol_1, vol_2, r2;
  if (lo) {
    vol_1 = cell_volume(i_r + 1, dr, dz);
    vol_2 = cell_volume(i_r + 3, dr, dz);
    r2 = (i_r + 1) * dr;
  } else {
    vol_1 = (radius.v > dr) ? cell_volume(i_r, dr, dz) : cyl_vol(dz, dr);
    r2 = (i_r + 0.5) * dr;
    vol_2 = cell_volume(i_r + 2, dr, dz);
  }
  D dz1, dz2;
  if (zhalf) {
    dz1 = (k_z + 1.5) * dz - longitude;
    dz2 = longitude - (k_z + 0.5) * dz;
  } else {
    dz1 = (k_z + 1) * dz - longitude;
    dz2 = longitude - k_z * dz;
  }
  GatherW out;
  out.ir = i_r;
  out.kz = k_z;
  // ring_term(F, dzx, ra, rb, vol) = F * pi * dzx * (rb^2 - ra^2) / vol
  D a_in = r2 * r2 - r1 * r1, a_out = r3 * r3 - r2 * r2;
  out.w[0] = kPi * dz1 * a_in / vol_1;
  out.w[1] = kPi * dz1 * a_out / vol_2;
  out.w[2] = kPi * dz2 * a_in / vol_1;
  out.w[3] = kPi * dz2 * a_out / vol_2;
  return out;
}

__device__ __forceinline__ D gather_d(const GridDesc &g, const double *F, D r, D z, bool lo, bool zhalf) {
  GatherW gw = gather_w(g, r, z, lo, zhalf);
  const double *row0 = F + (size_t)gw.ir * (size_t)g.nz + gw.kz;
  const double *row1 = row0 + g.nz;
  return gw.w[0] * row0[0] + gw.w[1] * row1[0] + gw.w[2] * row0[1] + gw.w[3] * row1[1];
}

constexpr int kAR = 0, kAPhi = 1, kAZ = 2;

__device__ __forceinline__ D dot3(const D *a, const D *b) {
  D res = cst(0.0);
  res = res + a[0] * b[0];
  res = res + a[1] * b[1];
  res = res + a[2] * b[2];
  return res;
}

// relativistic Boris (src/particles.cpp:1025-1150)
__device__ void boris_d(D q, D m, double dt, D e[3], D b[3], D v[3]) {
  D const1 = q * dt / (2 * m);
  for (int j = 0; j < 3; j++) e[j] = e[j] * const1;
  D bs = kMagnConst * const1;
  for (int j = 0; j < 3; j++) b[j] = b[j] * bs;
  D u[3], t[3];
  for (int j = 0; j < 3; j++) u[j] = (fabs(v[j].v) < kMnzl) ? cst(0.0) : v[j];
  D beta = dot3(u, u) / kC2;
  D gamma = 1 / dsqrt(1.0 - beta);
  for (int j = 0; j < 3; j++) u[j] = u[j] * gamma;
  for (int j = 0; j < 3; j++) u[j] = u[j] + e[j];
  gamma = drsqrt(1.0 + dot3(u, u) / kC2);
  for (int j = 0; j < 3; j++) b[j] = b[j] * gamma;
  D const2 = 2. / (1. + dot3(b, b));
  for (int j = 0; j < 3; j++) t[j] = u[j];
  u[0] = t[0] + const2 * ((t[1] - t[0] * b[2] + t[2] * b[0]) * b[2] - (t[2] + t[0] * b[1] - t[1] * b[0]) * b[1]);
  u[1] = t[1] + const2 * (-(t[0] + t[1] * b[2] - t[2] * b[1]) * b[2] + (t[2] + t[0] * b[1] - t[1] * b[0]) * b[0]);
  u[2] = t[2] + const2 * ((t[0] + t[1] * b[2] - t[2] * b[1]) * b[1] - (t[1] - t[0] * b[2] + t[2] * b[0]) * b[0]);
  for (int j = 0; j < 3; j++) u[j] = u[j] + e[j];
  gamma = drsqrt(1.0 + dot3(u, u) / kC2);
  for (int j = 0; j < 3; j++) v[j] = u[j] * gamma;
}

// Vay with the reference's scaling (src/particles.cpp:1152-1254)
__device__ void vay_d(D q, D m, double dt, D e[3], D b[3], D v[3]) {
  D const1 = q * dt / (2 * m);
  D s2 = 2 * const1;
  for (int j = 0; j < 3; j++) e[j] = e[j] * s2;
  D bs = kMagnConst * const1;
  for (int j = 0; j < 3; j++) b[j] = b[j] * bs;
  D u[3], t[3];
  for (int j = 0; j < 3; j++) u[j] = (fabs(v[j].v) < kMnzl) ? cst(0.0) : v[j];
  D beta = dot3(u, u) / kC2;
  D gamma = 1 / dsqrt(1.0 - beta);
  for (int j = 0; j < 3; j++) u[j] = u[j] * gamma;
  for (int j = 0; j < 3; j++) t[j] = u[j];
  for (int j = 0; j < 3; j++) b[j] = b[j] * s2;
  for (int j = 0; j < 3; j++) u[j] = u[j] + e[j];
  for (int j = 0; j < 3; j++) b[j] = b[j] * const1;
  gamma = drsqrt(1.0 + dot3(t, t) / kC2);
  u[0] = u[0] + gamma * (t[1] * b[2] - t[2] * b[1]);
  u[1] = u[1] + gamma * (t[2] * b[0] - t[0] * b[2]);
  u[2] = u[2] + gamma * (t[0] * b[1] - t[1] * b[0]);
  gamma = drsqrt(1.0 + dot3(u, u) / kC2);
  D alpha = 1. / gamma / gamma;
  D B2 = dot3(b, b);
  D sg = alpha - B2;
  D ub = dot3(u, b);
  D us2 = ub * ub;
  alpha = 1. / dsqrt(0.5 * (sg + dsqrt(sg * sg + 4. * (B2 + us2))));
  for (int j = 0; j < 3; j++) b[j] = b[j] * alpha;
  sg = 1. / (1. + dot3(b, b));
  alpha = dot3(u, b);
  t[0] = sg * (u[0] + alpha * b[0] + b[2] * u[1] - b[1] * u[2]);
  t[1] = sg * (u[1] + alpha * b[1] + b[0] * u[2] - b[2] * u[0]);
  t[2] = sg * (u[2] + alpha * b[2] + b[1] * u[0] - b[0] * u[1]);
  gamma = drsqrt(1.0 + dot3(t, t) / kC2);
  for (int j = 0; j < 3; j++) v[j] = t[j] * gamma;
}

__device__ __forceinline__ D ring(D F, D dzx, D ra, D rb, double vol) { return F * kPi * dzx * (rb * rb - ra * ra) / vol; }

// azimuthal_current_distribution, src/particles.cpp:688-784
template <class S>
__device__ void jphi_d(const GridDesc &g, S &sk, D q, D r, D z, D vphi) {
  const double dr = g.dr, dz = g.dz;
  int r_i = cell_number(r.v, dr), z_k = cell_number(z.v, dz);
  if (r_i < 0) r_i = 0;
  if (z_k < 0) z_k = 0;
  D r1 = r - 0.5 * dr;
  D r2 = cst((r_i + 0.5) * dr);
  D r3 = r + 0.5 * dr;
  D ro_v = q / (2. * kPi * dz * dr * r);
  double v_1 = (r.v > dr) ? cell_volume(r_i, dr, dz) : cyl_vol(dz, dr);
  double v_2 = cell_volume(r_i + 1, dr, dz);
  D dz1 = (z_k + 0.5) * dz - (z - 0.5 * dz);
  D dz2 = (z + 0.5 * dz) - (z_k + 0.5) * dz;
  sk.add(kAPhi, r_i, z_k, ring(ro_v, dz1, r1, r2, v_1) * vphi);
  sk.add(kAPhi, r_i + 1, z_k, ring(ro_v, dz1, r2, r3, v_2) * vphi);
  sk.add(kAPhi, r_i, z_k + 1, ring(ro_v, dz2, r1, r2, v_1) * vphi);
  sk.add(kAPhi, r_i + 1, z_k + 1, ring(ro_v, dz2, r2, r3, v_2) * vphi);
}

// (log(1+x) - x) / x without cancellation (series below |x| = 0.1)
__device__ __forceinline__ D m_of_d(D x) {
  if (fabs(x.v) < 0.1) {
    D s = cst(-1.0 / 12.0);
    const double c[] = {1.0 / 11.0, -0.1, 1.0 / 9.0, -0.125, 1.0 / 7.0, -1.0 / 6.0, 0.2, -0.25, 1.0 / 3.0, -0.5};
    for (double ck : c) s = ck + x * s;
    return x * s;
  }
  D l;
  l.v = log1p(x.v);
  for (int j = 0; j < kDN; j++) l.d[j] = x.d[j] / (1.0 + x.v);
  return (l - x) / x;
}

// simple_current_distribution, src/particles.cpp:333-474.  Values: the
// reference's expressions.  Derivatives: those of the same integrals written
// without cancellation in cell units (r = (i + a) dr, rho = i + a,
// x = drho / rho, M = (ln(1+x) - x) / x, N = -x / (1+x) - M):
//   J_z[i]   = q dzeta / (4 pi dr^2 dt) [ (1-a)(2i+a)/rho - drho/2 + i(i+1)/rho M ] / i
//   J_z[i+1] = q dzeta / (4 pi dr^2 dt) [ a(2i+1+a)/rho + drho/2 - i(i+1)/rho M ] / (i+1)
//   J_r[k]   = q / (2 pi dr dz dt) [ drho((1-b)/2 - dzeta/4) + i(i+1)/(2 rho) (drho (1-b)/rho_e + dzeta N) ] / (i+1/2)
//   J_r[k+1] = q / (2 pi dr dz dt) [ drho(b/2 + dzeta/4) + i(i+1)/(2 rho) (drho b/rho_e - dzeta N) ] / (i+1/2)
// (and the polynomial forms on the axis cell).  The reference's forms are
// differences of O(i) terms: their derivative loses ~1/x digits for nearly
// axial paths, which a relativistic beam's particles are.
template <class S>
__device__ void segment_d(const GridDesc &g, S &acc, D q, D radius_new, D longitude_new, D radius_old,
                          D longitude_old, int i_n, int k_n) {
  const double dr = g.dr, dz = g.dz, delta_t = g.dt;
  const double delta_r = radius_new.v - radius_old.v;
  const double delta_z = longitude_new.v - longitude_old.v;
  if ((fabs(delta_r) < kMnzl) || (fabs(delta_z) < kMnzl)) return;
  // values, as the reference computes them
  double vz0, vz1, vr0, vr1;
  {
    const double qv = q.v;
    double k = delta_r / delta_z;
    double b = radius_old.v;
    double lg = log((k * delta_z + b) / b);
    if (i_n >= 1) {
      double ssd = qv / (2 * kPi * (i_n * dr) * dr * dz * delta_t * 2 * dr);
      vz0 = ssd * (dr * delta_z - k * delta_z * delta_z / 2. - delta_z * b +
                   dr * dr / k * ((i_n + 0.5) * (i_n + 0.5) - 0.25) * lg);
      ssd = qv / (2 * kPi * ((i_n + 1) * dr) * dr * dz * delta_t * 2 * dr);
      vz1 = ssd * (k * delta_z * delta_z / 2. + delta_z * b + delta_z * dr +
                   dr * dr / k * (0.25 - (i_n + 0.5) * (i_n + 0.5)) * lg);
    } else {
      double ssd = qv / (2. * kPi * dr / 4. * dr * dz * delta_t * dr);
      vz0 = ssd * (dr * delta_z - k * delta_z * delta_z / 2. - delta_z * b);
      ssd = qv / (2 * kPi * dr * dr * dz * delta_t * 2 * dr);
      vz1 = ssd * (k * delta_z * delta_z / 2. + delta_z * dr + delta_z * b);
    }
    k = -delta_z / delta_r;
    const double r0 = (i_n + 0.5) * dr;
    const double r1 = radius_old.v;
    b = (k_n + 1.) * dz - longitude_old.v;
    const double ssd = qv / (2 * kPi * r0 * dr * dz * delta_t * dz);
    const double lr = log((radius_old.v + delta_r) / radius_old.v);
    vr0 = ssd * (r0 * k * delta_r + k / 2. * delta_r * (radius_old.v + delta_r / 2.) +
                 0.5 * delta_r * (b - k * (2 * r0 + r1)) +
                 delta_r * (b - k * r1) * (4 * r0 * r0 - dr * dr) / (8 * radius_old.v * (radius_old.v + delta_r)) +
                 (k * (r0 * r0 / 2. - dr * dr / 8.)) * lr);
    b = longitude_old.v - k_n * dz;
    vr1 = ssd * (-r0 * k * delta_r - k / 2. * delta_r * (radius_old.v + delta_r / 2.) +
                 0.5 * delta_r * (b + k * (2 * r0 + r1)) +
                 delta_r * (b + k * r1) * (4 * r0 * r0 - dr * dr) / (8 * radius_old.v * (radius_old.v + delta_r)) -
                 (k * (r0 * r0 / 2. - dr * dr / 8.)) * lr);
  }
  // derivatives, from the cancellation-free forms
  const double fi = (double)i_n;
  D a = radius_old / dr - fi;
  D bo = longitude_old / dz - (double)k_n;
  D drho = (radius_new - radius_old) / dr;
  D dzeta = (longitude_new - longitude_old) / dz;
  D jz0, jz1, jr0, jr1;
  if (i_n == 0) {
    jz0 = 8.0 * (1.0 - 0.5 * drho - a);
    jz1 = 0.5 * drho + 1.0 + a;
    jr0 = drho * (0.5 * (1.0 - bo) - 0.25 * dzeta) * 2.0;
    jr1 = drho * (0.5 * bo + 0.25 * dzeta) * 2.0;
  } else {
    D rs = fi + a;
    D re = rs + drho;
    D x = drho / rs;
    D M = m_of_d(x);
    D N = -(x / (1.0 + x)) - M;
    const double ii = fi * (fi + 1.0);
    jz0 = ((1.0 - a) * (2.0 * fi + a) / rs - 0.5 * drho + ii / rs * M) / fi;
    jz1 = (a * (2.0 * fi + 1.0 + a) / rs + 0.5 * drho - ii / rs * M) / (fi + 1.0);
    D cc = 0.5 * ii / rs;
    jr0 = (drho * (0.5 * (1.0 - bo) - 0.25 * dzeta) + cc * (drho * (1.0 - bo) / re + dzeta * N)) / (fi + 0.5);
    jr1 = (drho * (0.5 * bo + 0.25 * dzeta) + cc * (drho * bo / re - dzeta * N)) / (fi + 0.5);
  }
  D sz = q * dzeta / (4.0 * kPi * dr * dr * delta_t);
  D sr = q / (2.0 * kPi * dr * dz * delta_t);
  D out[4] = {sz * jz0, sz * jz1, sr * jr0, sr * jr1};
  out[0].v = vz0;
  out[1].v = vz1;
  out[2].v = vr0;
  out[3].v = vr1;
  acc.add(kAZ, i_n, k_n, out[0]);
  acc.add(kAZ, i_n + 1, k_n, out[1]);
  acc.add(kAR, i_n, k_n, out[2]);
  acc.add(kAR, i_n, k_n + 1, out[3]);
}

// strict_motion_weighting, src/particles.cpp:786-988
template <class S>
__device__ void strict_d(const GridDesc &g, S &acc, D q, D radius_new, D longitude_new, D radius_old,
                         D longitude_old) {
  const double dr = g.dr, dz = g.dz, delta_t = g.dt;
  int i_n = cell_number(radius_new.v, dr), k_n = cell_number(longitude_new.v, dz);
  int i_o = cell_number(radius_old.v, dr), k_o = cell_number(longitude_old.v, dz);
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

struct SegD {
  D rn, zn, ro, zo;
  int i, k;
};

// current_distribution, src/particles.cpp:480-685
template <class S>
__device__ void deposit_j_d(const GridDesc &g, S &acc, D q, D pr, D pz, D por, D poz) {
  const double dr = g.dr, dz = g.dz;
  int i_n = cell_number(pr.v, dr), k_n = cell_number(pz.v, dz);
  int i_o = cell_number(por.v, dr), k_o = cell_number(poz.v, dz);
  if (i_n < 0) i_n = 0;
  if (k_n < 0) k_n = 0;
  if (i_o < 0) i_o = 0;
  if (k_o < 0) k_o = 0;
  if (por.v == (i_o + 1) * dr) i_o = i_n;
  if (poz.v == (k_o + 1) * dz) k_o = k_n;
  if (pr.v == (i_n + 1) * dr) i_n = i_o;
  if (pz.v == (k_n + 1) * dz) k_n = k_o;
  int res_cell = abs(i_n - i_o) + abs(k_n - k_o);
  if ((fabs(pr.v - por.v) < kMnzl) || (fabs(pz.v - poz.v) < kMnzl)) {
    strict_d(g, acc, q, pr, pz, por, poz);
    return;
  }
  if (res_cell == 0) {  // the common case, without the segment list (which lives in scratch memory)
    segment_d(g, acc, q, pr, pz, por, poz, i_n, k_n);
    return;
  }
  SegD s[3];
  int ns = 0;
  if (res_cell == 1) {
    if ((i_n != i_o) && (k_n == k_o)) {
      if (por.v > (i_n + 1) * dr) {
        D a = (por - pr) / (poz - pz);
        D r_b = cst((i_n + 1) * dr);
        D z_b = pz + (r_b - pr) / a;
        s[0] = SegD{r_b, z_b, por, poz, i_n + 1, k_n};
        s[1] = SegD{pr, pz, r_b, z_b, i_n, k_n};
      } else {
        D a = (pr - por) / (pz - poz);
        D r_b = cst(i_n * dr);
        D z_b = poz + (r_b - por) / a;
        s[0] = SegD{r_b, z_b, por, poz, i_n - 1, k_n};
        s[1] = SegD{pr, pz, r_b, z_b, i_n, k_n};
      }
      ns = 2;
    } else if ((i_n == i_o) && (k_n != k_o)) {
      if (poz.v < k_n * dz) {
        D z_b = cst(k_n * dz);
        D a = (pr - por) / (pz - poz);
        D r_b = por + a * (z_b - poz);
        s[0] = SegD{r_b, z_b, por, poz, i_n, k_n - 1};
        s[1] = SegD{pr, pz, r_b, z_b, i_n, k_n};
      } else {
        D z_b = cst((k_n + 1) * dz);
        D a = (por - pr) / (poz - pz);
        D r_b = pr + a * (z_b - pz);
        s[0] = SegD{r_b, z_b, por, poz, i_n, k_n + 1};
        s[1] = SegD{pr, pz, r_b, z_b, i_n, k_n};
      }
      ns = 2;
    }
  } else if (res_cell == 2) {
    if (i_o < i_n) {
      if (k_o < k_n) {
        D a = (pr - por) / (pz - poz);
        D r1 = cst(i_n * dr);
        D z1 = poz + (r1 - por) / a;
        D z2 = cst(k_n * dz);
        D r2 = por + (z2 - poz) * a;
        if (z1.v < k_n * dz) {
          s[0] = SegD{r1, z1, por, poz, i_n - 1, k_n - 1};
          s[1] = SegD{r2, z2, r1, z1, i_n, k_n - 1};
          s[2] = SegD{pr, pz, r2, z2, i_n, k_n};
          ns = 3;
        } else if (z1.v > k_n * dz) {
          s[0] = SegD{r2, z2, por, poz, i_n - 1, k_n - 1};
          s[1] = SegD{r1, z1, r2, z2, i_n - 1, k_n};
          s[2] = SegD{pr, pz, r1, z1, i_n, k_n};
          ns = 3;
        }
      } else {
        D a = (pr - por) / (pz - poz);
        D r1 = cst(i_n * dr);
        D z1 = poz + (r1 - por) / a;
        D z2 = cst((k_n + 1) * dz);
        D r2 = por + -(poz - z2) * a;
        if (z1.v > (k_n + 1) * dz) {
          s[0] = SegD{r1, z1, por, poz, i_n - 1, k_n + 1};
          s[1] = SegD{r2, z2, r1, z1, i_n, k_n + 1};
          s[2] = SegD{pr, pz, r2, z2, i_n, k_n};
          ns = 3;
        } else if (z1.v < (k_n + 1) * dz) {
          s[0] = SegD{r2, z2, por, poz, i_n - 1, k_n + 1};
          s[1] = SegD{r1, z1, r2, z2, i_n - 1, k_n};
          s[2] = SegD{pr, pz, r1, z1, i_n, k_n};
          ns = 3;
        }
      }
    } else if (i_o > i_n) {
      if (k_o < k_n) {
        D a = (pr - por) / (pz - poz);
        D r1 = cst((i_n + 1) * dr);
        D z1 = poz + -(por - r1) / a;
        D z2 = cst(k_n * dz);
        D r2 = por - -(z2 - poz) * a;
        if (z1.v < (k_n)*dz) {
          s[0] = SegD{r1, z1, por, poz, i_n + 1, k_n - 1};
          s[1] = SegD{r2, z2, r1, z1, i_n, k_n - 1};
          s[2] = SegD{pr, pz, r2, z2, i_n, k_n};
          ns = 3;
        } else if (z1.v > (k_n)*dz) {
          s[0] = SegD{r2, z2, por, poz, i_n + 1, k_n - 1};
          s[1] = SegD{r1, z1, r2, z2, i_n + 1, k_n};
          s[2] = SegD{pr, pz, r1, z1, i_n, k_n};
          ns = 3;
        }
      } else if (k_o > k_n) {
        D a = (por - pr) / (poz - pz);
        D r1 = cst((i_n + 1) * dr);
        D z1 = pz + (r1 - pr) / a;
        D z2 = cst((k_n + 1) * dz);
        D r2 = pr + (z2 - pz) * a;
        if (z1.v > (k_n + 1) * dz) {
          s[0] = SegD{r1, z1, por, poz, i_n + 1, k_n + 1};
          s[1] = SegD{r2, z2, r1, z1, i_n, k_n + 1};
          s[2] = SegD{pr, pz, r2, z2, i_n, k_n};
          ns = 3;
        } else if (z1.v < (k_n + 1) * dz) {
          s[0] = SegD{r2, z2, por, poz, i_n + 1, k_n + 1};
          s[1] = SegD{r1, z1, r2, z2, i_n + 1, k_n};
          s[2] = SegD{pr, pz, r1, z1, i_n, k_n};
          ns = 3;
        }
      }
    }
  }
#pragma nounroll
  for (int t = 0; t < ns; t++) segment_d(g, acc, q, s[t].rn, s[t].zn, s[t].ro, s[t].zo, s[t].i, s[t].k);
}

// reflection_single / Bunch::reflection_single on the half-step point
__device__ __forceinline__ void walls_d(const GridDesc &g, bool is_bunch, D &x, D &z, D &v0, D &v2, bool &alive) {
  const double dr = g.dr, dz = g.dz;
  const double radius_wall = g.r_size - dr / 2., longitude_wall = g.z_size - dz / 2.;
  const double half_dr = dr / 2., half_dz = dz / 2.;
  if (is_bunch) {
    if (x.v > radius_wall) alive = false;
    if (z.v > longitude_wall) alive = false;
  } else {
    if (x.v > radius_wall) {
      x = radius_wall * 2. - x;
      v0 = -v0;
    }
    if (z.v > longitude_wall) {
      z = longitude_wall * 2. - z;
      v2 = -v2;
    }
  }
  if (x.v < half_dr) {
    x = dr - x;
    v0 = -v0;
  }
  if (z.v < half_dz) {
    z = dz - z;
    v2 = -v2;
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
  b.g0 = 1.0 / sqrt(1.0 - dot(b.u, b.u) / kC2);
  return b;
}
// adjoint of v from the adjoint of U = g0 u
__device__ __forceinline__ V3 boost_back(const Boost &b, V3 v, V3 lU) {
  const double s = b.g0 * b.g0 * b.g0 / kC2 * dot(lU, b.u);
  const V3 l = fma3(s, b.u, b.g0 * lU);
  return V3{fabs(v.x) < kMnzl ? 0.0 : l.x, fabs(v.y) < kMnzl ? 0.0 : l.y, fabs(v.z) < kMnzl ? 0.0 : l.z};
}
__device__ __forceinline__ double inv_gamma(V3 u) { return 1.0 / sqrt(1.0 + dot(u, u) / kC2); }
// adjoint of u added for an adjoint lg of g = inv_gamma(u)
__device__ __forceinline__ V3 inv_gamma_back(double g, V3 u, double lg, V3 l) {
  return fma3(-(g * g * g) / kC2 * lg, u, l);
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
  const double B2 = dot(h, h), ub = dot(up, h), sg = 1.0 + dot(up, up) / kC2 - B2;
  const double al = 1.0 / sqrt(0.5 * (sg + sqrt(sg * sg + 4. * (B2 + ub * ub))));
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
  const double B2 = dot(h, h), ub = dot(up, h), sg = 1.0 + dot(up, up) / kC2 - B2;
  const double root = sqrt(sg * sg + 4. * (B2 + ub * ub));
  const double al = 1.0 / sqrt(0.5 * (sg + root));
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
  w.ir = min(max(cell_number(r - 0.5 * g.dr, g.dr), 0), g.nr - 2);
  const double r1 = r - 0.5 * g.dr, r3 = r + 0.5 * g.dr, r2 = (w.ir + 1) * g.dr;
  const double p1 = kPi / cell_volume(w.ir + 1, g.dr, g.dz), p2 = kPi / cell_volume(w.ir + 3, g.dr, g.dz);
  w.in = p1 * (r2 * r2 - r1 * r1);
  w.out = p2 * (r3 * r3 - r2 * r2);
  w.din = -2.0 * p1 * r1;
  w.dout = 2.0 * p2 * r3;
  return w;
}
__device__ __forceinline__ RingW ring_own(const GridDesc &g, double r) {
  RingW w;
  w.ir = min(max(cell_number(r, g.dr), 0), g.nr - 2);
  const double r1 = r - 0.5 * g.dr, r3 = r + 0.5 * g.dr, r2 = (w.ir + 0.5) * g.dr;
  const double p1 = kPi / ((r > g.dr) ? cell_volume(w.ir, g.dr, g.dz) : cyl_vol(g.dz, g.dr));
  const double p2 = kPi / cell_volume(w.ir + 2, g.dr, g.dz);
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
  c.kz = min(max(cell_number(half ? z - 0.5 * g.dz : z, g.dz), 0), g.nz - 2);
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
// an LDS box of kR x kABK nodes per component (anchored one row and two
// columns below the block's smallest cell) and added to the grid once per
// block; stencils outside the box go to the grid directly.  A plasma block
// lies along one row.  A bunch block spans the bunch's radius: in four rows
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
__device__ __forceinline__ double jphi_back(const GridDesc &g, const double *L, double q, double w, double r, double z,
                                            double vphi, double &lr, double &lz, double &lvphi) {
  const double dr = g.dr, dz = g.dz;
  const int i = max(cell_number(r, dr), 0), k = max(cell_number(z, dz), 0);
  const double r1 = r - 0.5 * dr, r2 = (i + 0.5) * dr, r3 = r + 0.5 * dr;
  const double i1 = 1.0 / ((r > dr) ? cell_volume(i, dr, dz) : cyl_vol(dz, dr)), i2 = 1.0 / cell_volume(i + 1, dr, dz);
  const double d1 = (k + 0.5) * dz - (z - 0.5 * dz), d2 = (z + 0.5 * dz) - (k + 0.5) * dz;
  const double l00 = lam_at(g, L, i, k) * i1, l10 = lam_at(g, L, i + 1, k) * i2;
  const double l01 = lam_at(g, L, i, k + 1) * i1, l11 = lam_at(g, L, i + 1, k + 1) * i2;
  const double in = r2 * r2 - r1 * r1, out = r3 * r3 - r2 * r2;
  const double lo = l00 * d1 + l01 * d2, hi = l10 * d1 + l11 * d2;
  const double G = in * lo + out * hi;
  const double ir = 1.0 / r, K = q * ir / (2. * dz * dr);
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

// reverse of one straight piece inside cell (i, k), from the closed forms
// above segment_d: S = sum lambda_J J and its derivatives with respect to the
// piece's ends
struct PieceAdj {
  double s, rn, zn, ro, zo;
};
__device__ __forceinline__ PieceAdj segment_back(const GridDesc &g, const AdjGrid &lg, double q, double rn, double zn,
                                                 double ro, double zo, int i, int k) {
  const double dr = g.dr, dz = g.dz;
  PieceAdj o{0.0, 0.0, 0.0, 0.0, 0.0};
  if ((fabs(rn - ro) < kMnzl) || (fabs(zn - zo) < kMnzl)) return o;
  const double fi = (double)i, idr = 1.0 / dr, idz = 1.0 / dz;
  const double a = ro / dr - fi, b = zo / dz - (double)k, drho = (rn - ro) / dr, dzeta = (zn - zo) / dz;
  const double kz = q / (4.0 * kPi * dr * dr * g.dt), kr = q / (2.0 * kPi * dr * dz * g.dt);
  // lambda_J times the scales of the pairs (without the dzeta of J_z)
  double gz0 = kz * lam_at(g, lg.ljz, i, k), gz1 = kz * lam_at(g, lg.ljz, i + 1, k);
  double gr0 = kr * lam_at(g, lg.ljr, i, k), gr1 = kr * lam_at(g, lg.ljr, i, k + 1);
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
  o.rn = sdr * idr;
  o.ro = (sa - sdr) * idr;
  o.zn = sdz * idz;
  o.zo = (sb - sdz) * idz;
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

// reverse of the J_r / J_z deposit of the straight path (ro, zo) -> (rn, zn)
// (current_distribution, src/particles.cpp:480-685): the path is split at the
// radial face r = rb (met at z1) and the axial face z = zb (met at r2) that it
// crosses; with s the path parameter of the crossing, the adjoint of z1 goes
// to the ends as (1-s, s) along z and times -dz/dr along r, that of r2 likewise
__device__ __forceinline__ PieceAdj deposit_j_back(const GridDesc &g, const AdjGrid &lg, double q, double rn, double zn,
                                                   double ro, double zo) {
  const double dr = g.dr, dz = g.dz;
  int i_n = max(cell_number(rn, dr), 0), k_n = max(cell_number(zn, dz), 0);
  int i_o = max(cell_number(ro, dr), 0), k_o = max(cell_number(zo, dz), 0);
  if (ro == (i_o + 1) * dr) i_o = i_n;
  if (zo == (k_o + 1) * dz) k_o = k_n;
  if (rn == (i_n + 1) * dr) i_n = i_o;
  if (zn == (k_n + 1) * dz) k_n = k_o;
  const int di = i_n - i_o, dk = k_n - k_o, res = abs(di) + abs(dk);
  if ((fabs(rn - ro) < kMnzl) || (fabs(zn - zo) < kMnzl)) {
    StrictSink sk{&g, &lg, {0.0, 0.0, 0.0, 0.0, 0.0}};
    strict_d(g, sk, cst(q), seed(rn, 0), seed(zn, 1), seed(ro, 2), seed(zo, 3));
    return sk.o;
  }
  // pieces: ns, the crossings in order (first / second), the cells before the last
  int ns = 1, i0 = i_n, k0 = k_n, i1 = i_n, k1 = k_n;
  bool rad = false, axi = false, rfirst = false;
  double rb = 0.0, zb = 0.0, z1 = 0.0, r2 = 0.0;
  const double slope = (rn - ro) / (zn - zo);
  if (res == 1) {
    ns = 2;
    if (di != 0) {
      rad = rfirst = true;
      const bool up = !(ro > (i_n + 1) * dr);
      rb = (up ? i_n : i_n + 1) * dr;
      z1 = up ? zo + (rb - ro) / slope : zn + (rb - rn) / slope;
      i0 = up ? i_n - 1 : i_n + 1;
    } else {
      axi = true;
      const bool up = zo < k_n * dz;
      zb = (up ? k_n : k_n + 1) * dz;
      r2 = up ? ro + slope * (zb - zo) : rn + slope * (zb - zn);
      k0 = up ? k_n - 1 : k_n + 1;
    }
  } else if (res == 2) {
    // a path across a radial and an axial face; the other two-cell jumps are
    // too long for a step and are treated as the forward pass treats them
    const bool up = di > 0, right = dk > 0;
    if (di == 0 || (!up && dk == 0)) {
      ns = 0;
    } else {
      rad = axi = true;
      rb = (up ? i_n : i_n + 1) * dr;
      zb = (right ? k_n : k_n + 1) * dz;
      const bool from_new = !up && !right;
      z1 = from_new ? zn + (rb - rn) / slope : zo + (rb - ro) / slope;
      r2 = from_new ? rn + (zb - zn) * slope : ro + (zb - zo) * slope;
      ns = z1 == zb ? 0 : 3;
      rfirst = right ? z1 < zb : z1 > zb;
      i0 = up ? i_n - 1 : i_n + 1;
      k0 = right ? k_n - 1 : k_n + 1;
      i1 = rfirst ? i_n : i0;
      k1 = rfirst ? k0 : k_n;
    }
  } else if (res > 2) {
    ns = 0;
  }
  // the crossings in path order
  const double cr0 = rfirst ? rb : r2, cz0 = rfirst ? z1 : zb;
  const double cr1 = rfirst ? r2 : rb, cz1 = rfirst ? zb : z1;
  PieceAdj o{0.0, 0.0, 0.0, 0.0, 0.0};
  double c0r = 0.0, c0z = 0.0, c1r = 0.0, c1z = 0.0;  // adjoints of the crossings
#pragma nounroll
  for (int t = 0; t < ns; t++) {
    const bool first = t == 0, last = t == ns - 1;
    const PieceAdj p = segment_back(g, lg, q, last ? rn : first ? cr0 : cr1, last ? zn : first ? cz0 : cz1,
                                    first ? ro : t == 1 ? cr0 : cr1, first ? zo : t == 1 ? cz0 : cz1,
                                    last ? i_n : first ? i0 : i1, last ? k_n : first ? k0 : k1);
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
  if (rad) {
    const double l = rfirst ? c0z : c1z, s = (rb - ro) / (rn - ro), is = 1.0 / slope;
    o.zo += (1.0 - s) * l;
    o.zn += s * l;
    o.ro -= is * (1.0 - s) * l;
    o.rn -= is * s * l;
  }
  if (axi) {
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
  // the scales of the push's fields: q / m does not depend on w
  const double c1 = s.charge * g.dt / (2 * s.mass);
  const double es = VAY ? 2 * c1 : c1, bs = VAY ? kMagnConst * c1 * (2 * c1) * c1 : kMagnConst * c1;
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
    const PieceAdj p = deposit_j_back(g, lg, s.charge, r2, z2, r0, z0);
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
  lw += jphi_back(g, lg.ljphi, s.charge, w, r1, z1, v.y, lr1, lz1, lv.y);
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
  // the box anchor: the smallest cell of the block's living particles
  int ci = INT_MAX, ck = INT_MAX;
  if (live) {
    ci = max(cell_number(pt.r, g.dr), 0);
    ck = max(cell_number(pt.z, g.dz), 0);
  }
  block_min2(ci, ck);
  if (ci == INT_MAX) ci = ck = 0;
  for (int t = threadIdx.x; t < kSize; t += blockDim.x) box[t] = 0.0;
  __syncthreads();
  const Box b{box, ci - 1, ck - 2};
  if (live) adj_particle<VAY>(g, f, lg, s, i, pt, b);
  else if (i < s.n) s.lr[i] = s.lz[i] = s.lvr[i] = s.lvphi[i] = s.lvz[i] = 0.0;
  __syncthreads();
  double *const lf[kABComp] = {lg.ler, lg.lephi, lg.lez, lg.lhr, lg.lhphi, lg.lhz};
  for (int t = threadIdx.x; t < kSize; t += blockDim.x) {
    const double v = box[t];
    if (v == 0.0) continue;
    const int comp = t / (Box::kR * kABK), rem = t - comp * Box::kR * kABK;
    const int gi = b.bi + rem / kABK, gk = b.bk + rem % kABK;
    // nodes off the grid never receive a stencil (gather_w clamps its cell)
    if ((unsigned)gi < (unsigned)g.nr && (unsigned)gk < (unsigned)g.nz)
      unsafeAtomicAdd(lf[comp] + (size_t)gi * (size_t)g.nz + gk, v);
  }
}

// ------------------------------------------------ tangent-linear (forward mode)
// The same particle step in dual numbers, seeded with kDN tangent directions
// of the state, of the gathered fields and of the weight instead of unit
// vectors: the derivative parts of the outputs are the tangents of the new
// state and of every deposit (J-dot, scattered with atomics).  Together with
// the forward field updates applied to tangent grids this is the
// tangent-linear model of the loop, the exact transpose of what the adjoint
// above computes; <dphi/dw, dw> from the adjoint must equal the tangent of phi
// along dw to round-off (the dot-product test).

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
  double charge, mass;
  long long n;                          // slots
};

// deposit tangents: every contribution v at node (i, k) adds its derivative
// part (one per direction) to the tangent J grids, through an LDS box of kR x
// kK nodes per component and direction for the nodes around the block's
// smallest cell (a particle's 48 global atomics, those of a bunch all on the
// same few nodes, were most of the kernel)
template <bool BUNCH>
struct TlmSink {
  static constexpr int kR = BUNCH ? 16 : 4, kK = BUNCH ? 32 : 64, kSize = 3 * kDN * kR * kK;
  const GridDesc *g;
  TlmJ j;
  double *box;  // LDS
  int bi, bk;   // node of box[.][0][0]
  __device__ __forceinline__ void add(int comp, int i, int k, D v) {
    if ((unsigned)i >= (unsigned)g->nr || (unsigned)k >= (unsigned)g->nz) return;
    const int li = i - bi, lk = k - bk;
    if ((unsigned)li < (unsigned)kR && (unsigned)lk < (unsigned)kK) {
      double *q = box + (comp * kDN * kR + li) * kK + lk;
#pragma unroll
      for (int d = 0; d < kDN; d++)
        if (v.d[d] != 0.0) atomicAdd(q + d * kR * kK, v.d[d]);
      return;
    }
    const size_t p = (size_t)i * (size_t)g->nz + (size_t)k;
#pragma unroll
    for (int d = 0; d < kDN; d++) {
      double *J = comp == kAR ? j.jr[d] : comp == kAPhi ? j.jphi[d] : j.jz[d];
      if (v.d[d] != 0.0) unsafeAtomicAdd(J + p, v.d[d]);
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

// the gather of the tangent fields at the particle's (value) position: the
// gather is linear in the field, so its tangent along the field is the same
// weights applied to the tangent grid
__device__ __forceinline__ double gather_value(const GridDesc &g, const double *F, double r, double z, bool lo,
                                               bool zhalf) {
  GatherW gw = gather_w(g, cst(r), cst(z), lo, zhalf);
  const double *row0 = F + (size_t)gw.ir * (size_t)g.nz + gw.kz;
  const double *row1 = row0 + g.nz;
  return gw.w[0].v * row0[0] + gw.w[1].v * row1[0] + gw.w[2].v * row0[1] + gw.w[3].v * row1[1];
}

template <bool BUNCH, class Sink>
__device__ __forceinline__ void tlm_particle(const GridDesc &g, const AdjFields &f, const TlmFields &tf, Sink &sk,
                                             const TlmSpecies &s, int pusher, long long i, bool live,
                                             const AdjParticle &pt) {
  const long long n = s.n;
  if (!live) {
    // dead (or padding) slots keep zero tangents; a particle injected later
    // starts with zero tangents, as its injected state does not depend on w
#pragma unroll
    for (int d = 0; d < kDN; d++) s.tr[d * n + i] = s.tz[d * n + i] = s.tvr[d * n + i] = s.tvphi[d * n + i] =
        s.tvz[d * n + i] = 0.0;
    return;
  }
  auto dual = [&](double v, const double *t) {
    D x;
    x.v = v;
#pragma unroll
    for (int d = 0; d < kDN; d++) x.d[d] = t[d * n + i];
    return x;
  };
  D r = dual(pt.r, s.tr), z = dual(pt.z, s.tz);
  D v[3] = {dual(pt.vr, s.tvr), dual(pt.vphi, s.tvphi), dual(pt.vz, s.tvz)};
  D w = dual(pt.w, s.tw);
  D q = s.charge * w, m = s.mass * w;
  const D r_old = r, z_old = z;
  const double r0v = r.v, z0v = z.v;
  D e[3], h[3];
  e[0] = gather_d(g, f.er, r, z, true, false);
  e[1] = gather_d(g, f.ephi, r, z, false, false);
  e[2] = gather_d(g, f.ez, r, z, false, true);
  h[0] = gather_d(g, f.hhr, r, z, false, true);
  h[1] = gather_d(g, f.hhphi, r, z, true, true);
  h[2] = gather_d(g, f.hhz, r, z, true, false);
#pragma unroll
  for (int d = 0; d < kDN; d++) {
    e[0].d[d] += gather_value(g, tf.er[d], r0v, z0v, true, false);
    e[1].d[d] += gather_value(g, tf.ephi[d], r0v, z0v, false, false);
    e[2].d[d] += gather_value(g, tf.ez[d], r0v, z0v, false, true);
    h[0].d[d] += gather_value(g, tf.hhr[d], r0v, z0v, false, true);
    h[1].d[d] += gather_value(g, tf.hhphi[d], r0v, z0v, true, true);
    h[2].d[d] += gather_value(g, tf.hhz[d], r0v, z0v, true, false);
  }
  if (pusher == 1)
    vay_d(q, m, g.dt, e, h, v);
  else
    boris_d(q, m, g.dt, e, h, v);
  const double half_dt = g.dt / 2.;
  D x = r + v[0] * half_dt;
  D y = 0.0 + v[1] * half_dt;
  z = z + v[2] * half_dt;
  r = dsqrt(x * x + y * y);
  jphi_d(g, sk, q, r, z, v[1]);
  x = r + v[0] * half_dt;
  y = 0.0 + v[1] * half_dt;
  z = z + v[2] * half_dt;
  bool alive = true;
  walls_d(g, BUNCH, x, z, v[0], v[2], alive);
  D rr = dsqrt(x * x + y * y);
  D st = y / rr;
  r = rr;
  if (alive) {
    deposit_j_d(g, sk, q, r, z, r_old, z_old);
    D ct = dsqrt(1 - st * st);
    D u2 = ct * v[0] - st * v[1];
    D w2 = st * v[0] + ct * v[1];
    v[0] = u2;
    v[1] = w2;
  }
#pragma unroll
  for (int d = 0; d < kDN; d++) {
    const bool keep = alive;
    s.tr[d * n + i] = keep ? r.d[d] : 0.0;
    s.tz[d * n + i] = keep ? z.d[d] : 0.0;
    s.tvr[d * n + i] = keep ? v[0].d[d] : 0.0;
    s.tvphi[d * n + i] = keep ? v[1].d[d] : 0.0;
    s.tvz[d * n + i] = keep ? v[2].d[d] : 0.0;
  }
}

template <bool BUNCH, bool F32>
__global__ void __launch_bounds__(256) k_tlm_particles(GridDesc g, AdjFields f, TlmFields tf, TlmJ tj, TlmSpecies s,
                                                       int pusher) {
  using Sink = TlmSink<BUNCH>;
  __shared__ double box[Sink::kSize];
  const long long i = adj_slot<BUNCH>();
  AdjParticle pt;
  const bool live = i < s.n && adj_load<F32>(g, s.st, i, pt);
  int ci = INT_MAX, ck = INT_MAX;
  if (live) {
    ci = max(cell_number(pt.r, g.dr), 0);
    ck = max(cell_number(pt.z, g.dz), 0);
  }
  block_min2(ci, ck);
  if (ci == INT_MAX) ci = ck = 0;
  for (int t = threadIdx.x; t < Sink::kSize; t += blockDim.x) box[t] = 0.0;
  __syncthreads();
  Sink sk{&g, tj, box, ci - 1, ck - 2};
  if (i < s.n) tlm_particle<BUNCH>(g, f, tf, sk, s, pusher, i, live, pt);
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
  AdjSpecies s{state, lstate[0], lstate[1], lstate[2], lstate[3], lstate[4], lw, charge, mass, n};
  const dim3 grid((unsigned)((n + 255) / 256));
  using K = void (*)(GridDesc, AdjFields, AdjGrid, AdjSpecies);
  static const K kernels[8] = {k_adj_particles<false, false, false>, k_adj_particles<true, false, false>,
                               k_adj_particles<false, true, false>,  k_adj_particles<true, true, false>,
                               k_adj_particles<false, false, true>,  k_adj_particles<true, false, true>,
                               k_adj_particles<false, true, true>,   k_adj_particles<true, true, true>};
  hipLaunchKernelGGL(kernels[(pusher == 1) + 2 * (is_bunch != 0) + 4 * (state.cell != nullptr)], grid, dim3(256), 0, st,
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
  TlmSpecies s{state, tstate[0], tstate[1], tstate[2], tstate[3], tstate[4], tw, charge, mass, n};
  const dim3 grid((unsigned)((n + 255) / 256));
  using K = void (*)(GridDesc, AdjFields, TlmFields, TlmJ, TlmSpecies, int);
  static const K kernels[4] = {k_tlm_particles<false, false>, k_tlm_particles<true, false>,
                               k_tlm_particles<false, true>, k_tlm_particles<true, true>};
  hipLaunchKernelGGL(kernels[(is_bunch != 0) + 2 * (state.cell != nullptr)], grid, dim3(256), 0, st, g, f, tf, tj, s,
                     pusher);
}

void launch_tlm_objective(const GridDesc &g, const double *ez, double *const *const *tgrid, int k0, int k1,
                          double scale, double *phi5, hipStream_t st) {
  hipLaunchKernelGGL(k_tlm_objective, dim3(1), dim3(256), 0, st, g, ez, tgrid[0][kEZ], tgrid[1][kEZ],
                     tgrid[2][kEZ], tgrid[3][kEZ], k0, k1, scale, phi5);
}

}  // namespace pdp3
