// FP64 objective + gradient: the plain kernel of
// Minimizer::formFunctionAndGradient (minimizer.cpp:83-369).
//
//   k_density64  phase I  (:140-157; electrondensity.cpp:12-56): rho per
//                site, then F(rho), F'(rho) once per site.
//   k_grad64     phase II (:162-351): pair terms and gradient per site, the
//                per-site objective share, and a fixed-shape block reduction.
//   k_final_sum  per lattice, a fixed-order sum of its block partials -> f.
//
// Analytic mode evaluates each unordered pair once (k_dens_own64 ->
// k_dens_recv64 -> k_grad_own64 -> k_grad_recv64): the pair's owner computes
// both ends' shares and writes the partner's share into the partner's
// received slot, as the mixed path does.  These two owner kernels take the EAM
// functions from FP64 polynomial tables in LDS, built from the long-double closed
// forms (see "pair-once").  FD mode keeps the per-site
// full-list loop nest of the reference (every pair from both ends), since
// its derivatives are the reference's central differences per site.
//
// One lane per site over ELL rows: a wave holds 64 consecutive sites of one
// species, reads slot t of their rows as one coalesced load, and keeps the
// per-site sums in registers (no atomics, so results are bitwise
// reproducible).  Blocks map to lattices through b2l, so one launch serves a
// batch of uneven lattices.  The 12-point rule of quadrature.cpp:43-75 is used
// in its structured form: point (c, +-) of site i displaces r along axis c by
// +-sqrt(6) sigma_i, point (c, +-) of site j by -+sqrt(6) sigma_j.  The
// Gauss-Hermite rule (A2C_QUAD_GH3) has its own instances of the pair
// kernels; each instance skips the lattices of the other rule, and the
// per-site kernels apply the rule's factors (1/12 and sqrt(6), or 1).
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "eam64.hpp"
#include "fe_internal.hpp"
#include "pair_rows.hpp"

namespace a2c {
namespace {

constexpr int TB = SITE_BLOCK;
constexpr double QW = 1.0 / 12.0;             // 0.5/dim, quadrature.cpp:39
constexpr double SQ6 = 2.449489742783178098;  // sqrt(2)*sqrt(dim/2)
constexpr int GH3 = A2C_QUAD_GH3;
// Factors the per-site kernels apply to the pair sums: the 12-point sums are
// unweighted (weight 1/12) and their sigma terms carry r . e_c, a factor
// sqrt(6) short of d/dsigma; the Gauss-Hermite sums are complete.
template <int RULE> constexpr double rule_qw() { return RULE == GH3 ? 1.0 : QW; }
template <int RULE> constexpr double rule_sq() { return RULE == GH3 ? 1.0 : SQ6; }

__device__ __forceinline__ Site load_site(const double* __restrict__ X, int s) {
  const double4 v = *reinterpret_cast<const double4*>(X + 4 * (size_t)s);
  return {{v.x, v.y, v.z}, v.w};
}

// d = q_i - image(q_j): periodic axes shift q_j by L*rint((q_j - q_i)/L).  A
// listed pair is within rc < L/2 of an image, far from a rounding tie, so
// (q_j - q_i)*(1/L) picks the same image as the quotient at a fraction of
// the cost of an FP64 divide.
__device__ __forceinline__ void pair_vec(const LatDev& S, const Site& a, const Site& b, double d[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double qj = b.q[c];
    if (S.periodic[c]) qj = qj - S.box[c] * rint((qj - a.q[c]) * S.ibox[c]);
    d[c] = a.q[c] - qj;
  }
}
// the same with the geometry held in registers (pair-owner loops)
__device__ __forceinline__ void pair_vec(const Image& g, const Site& a, const Site& b, double d[3]) {
  image_vec(g, a.q, b.q, d);
}
template <int DM>
__device__ __forceinline__ double dF(bool pd, double rho, double eps) {
  if (DM == A2C_DERIV_FD) {
    return pd ? (eam::F_Pd(rho + eps) - eam::F_Pd(rho - eps)) / (2.0 * eps)
              : (eam::F_H(rho + eps) - eam::F_H(rho - eps)) / (2.0 * eps);
  }
  return pd ? eam::F_Pd_vd(rho).d : eam::F_H_vd(rho).d;
}

// Point p in 0..11: axis c = (p>>1)%3, sign = p&1 ? -1 : +1, owner = p<6 ? i : j.
__device__ __forceinline__ void point_r(int p, const double d[3], double ai, double aj, double r[3]) {
  const int c = (p >> 1) % 3;
  const double sg = (p & 1) ? -1.0 : 1.0;
  const double disp = (p < 6) ? sg * ai : -sg * aj;
  r[0] = d[0]; r[1] = d[1]; r[2] = d[2];
  r[c] += disp;
}

// Sum of g(|r|) over the nodes of one pair: unweighted over the 12 points, or
// weighted over the 27 Gauss-Hermite nodes (rule_qw completes either).
template <int RULE, class Fn>
__device__ __forceinline__ double pair_quad(const double d[3], double si, double sj, Fn g) {
  double acc = 0.0;
  if (RULE == GH3) {
    const double sd = sqrt(si * si + sj * sj);
#pragma unroll 1
    for (int k = 0; k < 27; ++k) {
      double z[3], w;
      gh_node(k, z, w);
      const double r0 = d[0] + sd * z[0], r1 = d[1] + sd * z[1], r2 = d[2] + sd * z[2];
      acc += w * g(sqrt(r0 * r0 + r1 * r1 + r2 * r2));
    }
  } else {
    const double ai = SQ6 * si, aj = SQ6 * sj;
#pragma unroll
    for (int p = 0; p < 12; ++p) {
      double r[3];
      point_r(p, d, ai, aj, r);
      acc += g(sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]));
    }
  }
  return acc;
}

// ---------------------------------------------------------------- density
template <int DM, int RULE>
__global__ __launch_bounds__(TB) void k_density64(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l,
                                                  double eps) {
  const int blk = xcd_block();
  const LatDev& S = lats[b2l[blk]];
  if (S.rule != RULE) return;  // the other rule's instance serves this lattice
  const int s = (blk - S.blk0) * TB + threadIdx.x;
  const int N = S.npd + S.nh;
  if (s >= N) return;
  const double* __restrict__ X = S.X;
  const double* __restrict__ xo = S.x;
  const bool pd = s < S.npd;
  const int row = pd ? s : s - S.npd;
  const Ell LP = pd ? S.pdpd : S.hpd;
  const Ell LH = pd ? S.pdh : S.hh;
  const Site a = load_site(X, s);
  constexpr double qw = rule_qw<RULE>();
  double rho = 0.0;
  const int np = LP.cnt[row];
  for (int t = 0; t < np; ++t) {
    const int j = LP.idx[(size_t)t * LP.rows + row];
    const Site b = load_site(X, j);
    double d[3];
    pair_vec(S, a, b, d);
    rho += pair_quad<RULE>(d, a.s, b.s, [](double r) { return eam::f_Pd(r); }) * qw;
  }
  const int nhn = LH.cnt[row];
  for (int t = 0; t < nhn; ++t) {
    const int h = LH.idx[(size_t)t * LH.rows + row];
    const Site b = load_site(X, S.npd + h);
    double d[3];
    pair_vec(S, a, b, d);
    rho += xo[h] * pair_quad<RULE>(d, a.s, b.s, [](double r) { return eam::f_H(r); }) * qw;
  }
  S.rho[s] = rho;
  const double F = pd ? eam::F_Pd(rho) : eam::F_H(rho);
  S.Fp[s] = dF<DM>(pd, rho, eps);
  S.emb[s] = pd ? F : xo[row] * F;
}

// ---------------------------------------------------------------- gradient
// Pair kinds: 0 Pd-Pd, 1 Pd-H (site Pd), 2 H-Pd (site H), 3 H-H.
template <int DM, int KIND>
__device__ __forceinline__ void pair_point(double r, double Fi, double Fj, double eps, double& phi, double& c) {
  if (DM == A2C_DERIV_FD) {
    auto fd = [&](auto g) { return (g(r + eps) - g(r - eps)) / (2.0 * eps); };
    if (KIND == 0) {
      const double fpd = fd([](double x) { return eam::f_Pd(x); });
      phi = eam::phi_Pd(r);
      c = (Fi + Fj) * fpd + fd([](double x) { return eam::phi_Pd(x); });
    } else if (KIND == 1 || KIND == 2) {
      const double fpd = fd([](double x) { return eam::f_Pd(x); });
      const double fh = fd([](double x) { return eam::f_H(x); });
      phi = eam::phi_morse<0>(r);
      const double dph = fd([](double x) { return eam::phi_morse<0>(x); });
      c = (KIND == 1) ? Fi * fh + Fj * fpd + dph : Fi * fpd + Fj * fh + dph;
    } else {
      const double fh = fd([](double x) { return eam::f_H(x); });
      phi = eam::phi_morse<1>(r);
      c = (Fi + Fj) * fh + fd([](double x) { return eam::phi_morse<1>(x); });
    }
  } else {
    if (KIND == 0) {
      const eam::VD f = eam::f_Pd_vd(r);
      const eam::VD ph = eam::phi_Pd_vd(r, f);
      phi = ph.v;
      c = (Fi + Fj) * f.d + ph.d;
    } else if (KIND == 1 || KIND == 2) {
      const eam::VD f = eam::f_Pd_vd(r);
      const eam::VD h = eam::f_H_vd(r);
      const eam::VD ph = eam::phi_morse_vd<0>(r);
      phi = ph.v;
      c = (KIND == 1) ? Fi * h.d + Fj * f.d + ph.d : Fi * f.d + Fj * h.d + ph.d;
    } else {
      const eam::VD h = eam::f_H_vd(r);
      const eam::VD ph = eam::phi_morse_vd<1>(r);
      phi = ph.v;
      c = (Fi + Fj) * h.d + ph.d;
    }
  }
}

// Accumulate one neighbor pair: energy (phi summed over points), q-gradient
// and sigma-gradient (12-point rule: r . xi1 is nonzero only on the six
// points of site i; Gauss-Hermite rule: sum of w (c/|r|) (r . z) sigma_i/s).
template <int DM, int KIND, int RULE>
__device__ __forceinline__ void pair_accum(const double d[3], double si, double sj, double Fi, double Fj,
                                           double eps, double& e, double g[3], double& gs) {
  double pe = 0.0, px = 0.0, py = 0.0, pz = 0.0, ps = 0.0;
  if (RULE == GH3) {
    const double sd = sqrt(si * si + sj * sj);
#pragma unroll 1
    for (int k = 0; k < 27; ++k) {
      double z[3], w;
      gh_node(k, z, w);
      const double r[3] = {d[0] + sd * z[0], d[1] + sd * z[1], d[2] + sd * z[2]};
      const double rn = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
      double phi, c;
      pair_point<DM, KIND>(rn, Fi, Fj, eps, phi, c);
      pe += w * phi;
      const double u = w * c / rn;
      px += u * r[0];
      py += u * r[1];
      pz += u * r[2];
      ps += u * (r[0] * z[0] + r[1] * z[1] + r[2] * z[2]);
    }
    e += pe;
    g[0] += px; g[1] += py; g[2] += pz;
    gs += ps * (si / sd);
    return;
  }
  const double ai = SQ6 * si, aj = SQ6 * sj;
#pragma unroll 1  // rolled, as in pair_both
  for (int p = 0; p < 12; ++p) {
    double r[3];
    point_r(p, d, ai, aj, r);
    const double rn = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
    double phi, c;
    pair_point<DM, KIND>(rn, Fi, Fj, eps, phi, c);
    pe += phi;
    const double u = c / rn;
    px += u * r[0];
    py += u * r[1];
    pz += u * r[2];
    if (p < 6) {
      const int ax = (p >> 1) % 3;
      ps += ((p & 1) ? -u : u) * r[ax];  // (c/|r|) r . xi1 / sqrt(3)
    }
  }
  e += pe;
  g[0] += px; g[1] += py; g[2] += pz;
  gs += ps;
}

template <int DM, int RULE>
__global__ __launch_bounds__(TB) void k_grad64(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l,
                                               double eps) {
  __shared__ double red[TB];
  const int blk = xcd_block();
  const LatDev& S = lats[b2l[blk]];
  if (S.rule != RULE) return;  // whole block: the other rule's instance serves this lattice
  const int lb = blk - S.blk0;
  const int s = lb * TB + threadIdx.x;
  const int N = S.npd + S.nh;
  double fs = 0.0;
  if (s < N) {
    const double* __restrict__ X = S.X;
    const double* __restrict__ xo = S.x;
    const double* __restrict__ Fp = S.Fp;
    const bool pd = s < S.npd;
    const int row = pd ? s : s - S.npd;
    const Ell LP = pd ? S.pdpd : S.hpd;
    const Ell LH = pd ? S.pdh : S.hh;
    const Site a = load_site(X, s);
    const double Fi = Fp[s];
    const double xi = pd ? 1.0 : xo[row];
    double ePd = 0.0, eH = 0.0, g[3] = {0.0, 0.0, 0.0}, gs = 0.0;
    const int np = LP.cnt[row];
    for (int t = 0; t < np; ++t) {
      const int j = LP.idx[(size_t)t * LP.rows + row];
      const Site b = load_site(X, j);
      double d[3];
      pair_vec(S, a, b, d);
      if (pd) pair_accum<DM, 0, RULE>(d, a.s, b.s, Fi, Fp[j], eps, ePd, g, gs);
      else pair_accum<DM, 2, RULE>(d, a.s, b.s, Fi, Fp[j], eps, ePd, g, gs);
    }
    const int nhn = LH.cnt[row];
    for (int t = 0; t < nhn; ++t) {
      const int h = LH.idx[(size_t)t * LH.rows + row];
      const Site b = load_site(X, S.npd + h);
      double d[3];
      pair_vec(S, a, b, d);
      const double xh = xo[h];
      double e1 = 0.0, g1[3] = {0.0, 0.0, 0.0}, gs1 = 0.0;
      if (pd) pair_accum<DM, 1, RULE>(d, a.s, b.s, Fi, Fp[S.npd + h], eps, e1, g1, gs1);
      else pair_accum<DM, 3, RULE>(d, a.s, b.s, Fi, Fp[S.npd + h], eps, e1, g1, gs1);
      eH += xh * e1;
      g[0] += xh * g1[0]; g[1] += xh * g1[1]; g[2] += xh * g1[2];
      gs += xh * gs1;
    }
    // V share of site s: embedding + half of every pair (minimizer.cpp:169-286)
    constexpr double qw = rule_qw<RULE>(), sq = rule_sq<RULE>();
    const double V = S.emb[s] + 0.5 * qw * xi * (ePd + eH);
    const double T = S.T;
    const double sc = qw * xi / T;
    double* __restrict__ G = S.G;
    G[4 * (size_t)s + 0] = sc * g[0];
    G[4 * (size_t)s + 1] = sc * g[1];
    G[4 * (size_t)s + 2] = sc * g[2];
    G[4 * (size_t)s + 3] = sq * sc * gs - 3.0 * KB * xi / a.s;
    fs = V / T - 3.0 * KB * xi * log(a.s);
  }
  red[threadIdx.x] = fs;
  __syncthreads();
#pragma unroll
  for (int w = TB / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) S.part[lb] = red[0];
}

// ================================================================ pair-once
// The nodes of a pair one at a time, for the pairs that leave the tables:
// |r| of node k, its displacement z and its weight w (1 in the 12-point rule).
template <int RULE>
struct Closed {
  static constexpr int N = RULE == GH3 ? 27 : 12;
  double d[3], ai, aj, sd;
  __device__ __forceinline__ Closed(const double* dd, double si, double sj)
      : d{dd[0], dd[1], dd[2]}, ai(SQ6 * si), aj(SQ6 * sj), sd(sqrt(fma(si, si, sj * sj))) {}
  __device__ __forceinline__ double node(int k, double z[3], double& w) const {
    if (RULE == GH3) {
      gh_node(k, z, w);
#pragma unroll
      for (int c = 0; c < 3; ++c) z[c] *= sd;
    } else {
      w = 1.0;
      const int ax = (k >> 1) % 3;
      const double a = (k & 1 ? -1.0 : 1.0) * (k < 6 ? ai : -aj);
#pragma unroll
      for (int c = 0; c < 3; ++c) z[c] = c == ax ? a : 0.0;
    }
    const double r0 = d[0] + z[0], r1 = d[1] + z[1], r2 = d[2] + z[2];
    return sqrt(r0 * r0 + r1 * r1 + r2 * r2);
  }
};

// The owner passes read the EAM functions from polynomial tables.  The Pd functions
// stand on a uniform grid in s = |r|^2 (a node's coordinate is one addition, and
// dE/ds = (dE/dr) / (2 |r|) is what the gradient needs: no square root per
// node); h = 0.5025 / 13 puts their switch radii 5.0 and 5.05 A on grid nodes (25
// and 25.5025 A^2), and the rows reach past 36 A^2.  phi_PdH and phi_HH have rows
// in r, 1/40 A apart: exponentials are steepest at short distances, where steps
// in s are the longest in r; their other switch radius 5.35 A is a node of that
// grid; and a node of an H pair has r at hand from f_H.  A row is a polynomial in
// u in [0, 1): f_Pd (degree 7, density pass) and its slope (degree 7) interpolated
// at the Chebyshev points, the pair functions (phi_Pd degree 8, phi_PdH and phi_HH
// 7) as the integral of the interpolant of their slope, so that value and slope
// belong together.  The degrees are the lowest whose interpolation errors stay
// below the FP64 roundings of the closed forms: part of the Pd functions falls as
// e^{-51.6 (r - 5)} beyond 5.0 A, where degree 5 left 5e-12 of slopes of 0.08, and
// phi_HH in s 2e-11 at 2 A and 1.7e-9 across 5.35 A; now below 1e-15 and 1e-14
// (tests/test_pass_tables.py holds every function).  Row pitches are 16-byte
// multiples that spread a wave's rows over 16 bank groups (8 doubles: 4); the
// tables fill 158 of the 160 KB of LDS (one workgroup per CU).  f_H = 11.0025
// exp(-1.30927 |r|) is computed instead (exp2 by a 256-entry table and a degree-4
// polynomial): ~25 FP64 instructions on four SIMDs cost no more than a row, and the
// two pipes work side by side.
// A node's coordinate is x = SINV s + SB; the rows are built on the grid that these
// two doubles define (rounded apart, the grid would be 4e-15 off: 5e-14 of a slope
// at 1 A).
constexpr double SINV = 13.0 / 0.5025, SB = 635 - 25.5025 * SINV, SH = 1.0 / SINV, S0 = -SB / SINV;
constexpr double SLO = 1.0, SHI = 36.0;  // nodes the tables serve: [1, 6) A
constexpr int SNT = 908;                 // rows in s
static_assert(S0 < 1.0 && S0 + (SNT - 1) * SH > 36.0, "the grid covers [1, 36] A^2");
constexpr double RH = 1.0 / 40.0, RINV = 40.0, RB = -39.0;
constexpr int RNT = 202;                 // rows in r, the first at 39/40 A
static_assert((-RB + RNT - 0.5) * RH > 6.0, "the grid covers [1, 6] A");
constexpr int FD = 7, FP = 10;           // f_Pd rows: degree, pitch
constexpr int GD = 7, PHD = 8, GP = 18;  // f_Pd' (c0..c7) and phi_Pd (from 8) rows: degrees, common pitch
constexpr int RD = 7, RP = 18;           // phi_PdH and phi_HH (from 8) rows
constexpr int EXPN = 256;                // 2^(i / 256)
// offsets in doubles; each pass stages a contiguous part
constexpr int S_FPD = 0, S_PD = S_FPD + SNT * FP, S_PH = S_PD + SNT * GP, S_EXP = S_PH + RNT * RP;
constexpr int S_SIZE = S_EXP + EXPN;
static_assert(8 * (S_SIZE - S_PD) <= 160 << 10, "the gradient pass's tables fit the LDS");

struct SPos {
  int k;
  double u;
};
A2C_HD SPos s_pos(double x) { return {(int)x, eam::fract(x)}; }
A2C_HD double s_of(double x) { return fma(x, SH, S0); }
template <int P>
A2C_HD const double* row_at(const double* tab, int k) { return tab + eam::mul24(k, P); }
// D + 1 coefficients of a row (16-byte aligned), as 16-byte reads
template <int D>
struct Coef {
  double c[D + 1];
  A2C_HD explicit Coef(const double* p) {
#pragma unroll
    for (int j = 0; j < D; j += 2) {
      const double2 v = *reinterpret_cast<const double2*>(p + j);
      c[j] = v.x;
      c[j + 1] = v.y;
    }
    if (D % 2 == 0) c[D] = p[D];
  }
};
template <int D>
A2C_HD double poly(const double* row, double u) {
  const Coef<D> q(row);
  double v = q.c[D];
#pragma unroll
  for (int j = D - 1; j >= 0; --j) v = fma(v, u, q.c[j]);
  return v;
}
// value and d/du
template <int D>
A2C_HD void poly_vd(const double* row, double u, double& v, double& d) {
  const Coef<D> q(row);
  v = fma(q.c[D], u, q.c[D - 1]);
  d = fma(q.c[D], u, v);
#pragma unroll
  for (int j = D - 2; j >= 1; --j) {
    v = fma(v, u, q.c[j]);
    d = fma(d, u, v);
  }
  v = fma(v, u, q.c[0]);
}
// phi_PdH (tab: its rows) or phi_HH (8 beyond) at r, and d/du
A2C_HD void phi_r(const double* tab, double r, double& v, double& d) {
  const double y = fma(r, RINV, RB);
  poly_vd<RD>(row_at<RP>(tab, (int)y), eam::fract(y), v, d);
}
A2C_HD long long double_bits(double x) {
  long long b;
  __builtin_memcpy(&b, &x, sizeof b);
  return b;
}
// 1/sqrt(x): the hardware estimate y (relative error below 2^-20), then one
// step of y <- y (1 + e/2 + 3 e^2 / 8), e = 1 - x y^2 (third order).
A2C_HD double rsqrt3(double x) {
  const double y = eam::rsq_est(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}
// f_H / 11.0025 = 2^(E / 256), E = 256 log2(e) ln(f_H / 11.0025), at s = r^2, with r
// and 1/r; sl = f_H' / (-1.30927 11.0025).  n = rint(E) picks 2^(n/256) from the
// table, the remainder f in [-1/2, 1/2] goes through the series of 2^(f/256) (next
// term 4e-17).  E = K r up to 5.35 A and K2 r + B2 on the tail beyond, which
// potential.cpp gives another amplitude (5e-14 off at 5.35 A) and decay (2.5e-11): 256
// log2(e) ln(0.009986990526578 / 11.0025 exp(5.35 FH_K2)) is B2.  The choice costs
// 7% of an evaluation, so a wave's pairs make it (TAIL) only if one of them has
// a node there (40^3 cells: 1069 us without it, 1142 with it in every pair).
constexpr double FH_K = -1.30927, FH_K2 = -0.013075667086408 / 0.009986990526578;
template <bool TAIL>
A2C_HD double fH_s(const double* exptab, double s, double& r, double& ri, double& sl) {
  constexpr double C = 1.4426950408889634074 * EXPN, MAGIC = 6755399441055744.0;
  constexpr double K = FH_K * C, K2 = FH_K2 * C, B2 = -6.42743196697137263e-8;
  constexpr double L1 = 0.69314718055994530942 / EXPN;
  ri = rsqrt3(s);
  r = s * ri;
  const bool tail = TAIL && r > 5.35;
  const double k = tail ? K2 : K;
  const double t = fma(r, k, MAGIC);
  const int n = (int)(unsigned)double_bits(t);
  const double f = fma(r, k, (tail ? B2 : 0.0) - (t - MAGIC));
  const double p = f * fma(f, fma(f, fma(f, L1 * L1 * L1 * L1 / 24.0, L1 * L1 * L1 / 6.0), L1 * L1 / 2.0), L1);
  const double T = ldexp(exptab[n & (EXPN - 1)], n >> 8), v = fma(T, p, T);
  sl = v * (tail ? FH_K2 / FH_K : 1.0);
  return v;
}

// Table coordinates of one pair: 12-point rule (site e's nodes have
// x = xb +- g d_c with g = 2 a / h, see pair_both) and Gauss-Hermite rule
// (x = x0 + n1 |a|^2 + a . t).  inside(): every node lies in [1, 6) A; written in
// explicit fma, so that the passes that ask get the same answer.
struct Nodes12 {
  double xi, xj, gi, gj, lo, hi;
  __device__ __forceinline__ Nodes12(const double d[3], double ai, double aj) {
    const double D2 = fma(d[0], d[0], fma(d[1], d[1], d[2] * d[2]));
    const double bi = fma(ai, ai, D2), bj = fma(aj, aj, D2);
    const double ei = 2.0 * ai, ej = 2.0 * aj;
    const double m = fmax(fmax(fabs(d[0]), fabs(d[1])), fabs(d[2]));
    lo = fmin(fma(-fabs(ei), m, bi), fma(-fabs(ej), m, bj));
    hi = fmax(fma(fabs(ei), m, bi), fma(fabs(ej), m, bj));
    xi = fma(bi, SINV, SB);
    xj = fma(bj, SINV, SB);
    gi = ei * SINV;
    gj = ej * SINV;
  }
};
struct Nodes27 {
  double x0, n1, t[3], lo, hi;
  __device__ __forceinline__ Nodes27(const double d[3], double sd) {
    const double D2 = fma(d[0], d[0], fma(d[1], d[1], d[2] * d[2]));
    const double s3 = 3.0 * sd * sd, tt = 2.0 * GH_Z * sd;
    lo = hi = D2;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      lo += fmin(fma(-tt, fabs(d[c]), s3), 0.0);
      hi += fma(tt, fabs(d[c]), s3);
      t[c] = tt * SINV * d[c];
    }
    x0 = fma(D2, SINV, SB);
    n1 = s3 * SINV;
  }
};
__device__ __forceinline__ bool inside(double lo, double hi) { return lo >= SLO && hi < SHI; }
// some pair of the wave has a node on f_H's tail (a margin over the roundings of hi and r)
__device__ __forceinline__ bool on_tail(double hi) { return __ballot(hi > 5.35 * 5.35 - 1e-9) != 0; }

// densities at one node inside the tables
template <bool WANT_PD, bool WANT_H, bool TAIL>
__device__ __forceinline__ void node_dens(const double* tab, const double* exptab, double x, double& fpd, double& fh) {
  if (WANT_PD) {
    const SPos p = s_pos(x);
    fpd = poly<FD>(row_at<FP>(tab, p.k), p.u);
  }
  if (WANT_H) {
    double r, ri, sl;
    fh = fH_s<TAIL>(exptab, s_of(x), r, ri, sl);
  }
}

// Sums of f_Pd and f_H over the nodes of one pair in closed form.
template <int RULE>
__device__ __forceinline__ double2 closed_dens(const double d[3], double si, double sj) {
  const Closed<RULE> q(d, si, sj);
  double sp = 0.0, sh = 0.0;
#pragma unroll 1
  for (int k = 0; k < Closed<RULE>::N; ++k) {
    double z[3], w;
    const double r = q.node(k, z, w);
    sp += w * eam::f_Pd(r);
    sh += w * eam::f_H(r);
  }
  return make_double2(sp, sh);
}

// Sums over a pair's nodes of f_Pd and of f_H / 11.0025, as wanted.
template <bool WP, bool WH, bool TAIL>
__device__ __forceinline__ void dens_sums27(const double* tab, const double* exptab, const Nodes27& q, double& sp,
                                            double& sh) {
#pragma unroll 1
  for (int a2 = -1; a2 <= 1; ++a2) {
#pragma unroll 1
    for (int a1 = -1; a1 <= 1; ++a1) {
      const double xb = q.x0 + q.n1 * (double)(a2 * a2 + a1 * a1) + ((double)a2 * q.t[2] + (double)a1 * q.t[1]);
      const double w = (a2 ? 1.0 : 4.0) * (a1 ? 1.0 : 4.0);
      double pp = 0.0, ph = 0.0;
#pragma unroll
      for (int a0 = -1; a0 <= 1; ++a0) {
        double fp = 0.0, fh = 0.0;
        node_dens<WP, WH, TAIL>(tab, exptab, a0 ? xb + q.n1 + a0 * q.t[0] : xb, fp, fh);
        pp += a0 ? fp : 4.0 * fp;
        ph += a0 ? fh : 4.0 * fh;
      }
      sp = fma(w, pp, sp);
      sh = fma(w, ph, sh);
    }
  }
  sp *= 1.0 / 216.0;
  sh *= 1.0 / 216.0;
}
template <bool WP, bool WH, bool TAIL>
__device__ __forceinline__ void dens_sums12(const double* tab, const double* exptab, const Nodes12& q,
                                            const double d[3], double& sp, double& sh) {
  double d0 = d[0], d1 = d[1], d2 = d[2];
  constexpr int UN = TAIL ? 1 : 3;  // the rare instance would spill unrolled
#pragma unroll UN
  for (int c = 0; c < 3; ++c) {
    const double ti = q.gi * d0, tj = q.gj * d0;
    const double x[4] = {q.xi + ti, q.xi - ti, q.xj - tj, q.xj + tj};
    constexpr int UK = TAIL ? 1 : 4;
#pragma unroll UK
    for (int k = 0; k < 4; ++k) {
      double fp = 0.0, fh = 0.0;
      node_dens<WP, WH, TAIL>(tab, exptab, k == 0 ? x[0] : k == 1 ? x[1] : k == 2 ? x[2] : x[3], fp, fh);
      if (WP) sp += fp;
      if (WH) sh += fh;
    }
    d0 = d1;
    d1 = d2;
  }
}

// Sums over a pair's nodes of the density of the neighbor's species (mine) and
// of this site's species (theirs); NB_H / ME_H: neighbor / this site is an H
// site.  False, and zeros, if a node lies outside the tables.
template <int RULE, bool NB_H, bool ME_H>
__device__ __forceinline__ bool pair_dens(const double* tab, const double* exptab, const double d[3], double si,
                                          double sj, double& mine, double& theirs) {
  constexpr bool WP = !NB_H || !ME_H, WH = NB_H || ME_H;
  double sp = 0.0, sh = 0.0;
  bool in;
  if (RULE == GH3) {
    const Nodes27 q(d, sqrt(fma(si, si, sj * sj)));
    in = inside(q.lo, q.hi);
    if (in) {
      if (WH && on_tail(q.hi)) dens_sums27<WP, WH, true>(tab, exptab, q, sp, sh);
      else dens_sums27<WP, WH, false>(tab, exptab, q, sp, sh);
    }
  } else {
    const Nodes12 q(d, SQ6 * si, SQ6 * sj);
    in = inside(q.lo, q.hi);
    if (in) {
      if (WH && on_tail(q.hi)) dens_sums12<WP, WH, true>(tab, exptab, q, d, sp, sh);
      else dens_sums12<WP, WH, false>(tab, exptab, q, d, sp, sh);
    }
  }
  sh *= 11.0025;
  mine = NB_H ? sh : sp;
  theirs = ME_H ? sh : sp;
  return in;
}

// The pairs of a row that leave the tables, after its other pairs: the closed
// forms hold ~190 registers and would cost every pair its waves if they stood
// in its loop.
template <bool NB_H, class Fn>
__device__ __forceinline__ void far_pairs(const Ell& L, const OwnerLane& ln, int K, const LatDev& S, Fn fn) {
  const int n = L.ocnt[ln.row];
  for (int t = ln.ph; t < n; t += K) {
    const size_t e = (size_t)t * L.rows + ln.row;
    fn(L.oj[e], L.orv[e], (NB_H ? S.npd : 0) + L.oj[e]);
  }
}
template <int RULE>
__device__ __forceinline__ bool pair_inside(const double d[3], double si, double sj) {
  if (RULE == GH3) {
    const Nodes27 n(d, sqrt(fma(si, si, sj * sj)));
    return inside(n.lo, n.hi);
  }
  const Nodes12 n(d, SQ6 * si, SQ6 * sj);
  return inside(n.lo, n.hi);
}

struct Pair64 {
  double d[3], s;
};
template <int RULE, bool BY_SITE, bool NB_H, bool ME_H>
__device__ __forceinline__ void dens_list(const double* tab, const double* exptab, const LatDev& S,
                                          const OwnerLane& ln, const Site& a, const Image& img, double wme,
                                          double& rho) {
  const Ell& L = ME_H ? (NB_H ? S.hh : S.hpd) : (NB_H ? S.pdh : S.pdpd);
  const Ell& P = ME_H ? (NB_H ? S.hh : S.pdh) : (NB_H ? S.hpd : S.pdpd);  // partner rows
  A2C_GLOBAL double* __restrict__ share = gmem(reinterpret_cast<double*>(P.rbuf));
  const size_t prows = P.rows;
  bool far = false;
  owned_pairs<NB_H, BY_SITE>(
      L, ln, S.kl64, S, [](int) { return 0.0f; },
      [&](const Site& b) {
        Pair64 p;
        pair_vec(img, a, b, p.d);
        p.s = b.s;
        return p;
      },
      [&](const Pair64& p, float, double wj, int jl, int rv) {
        double mine, theirs;
        far |= !pair_dens<RULE, NB_H, ME_H>(tab, exptab, p.d, a.s, p.s, mine, theirs);
        rho += wj * mine;
        // shares leave weighted by the sender's occupancy
        share[(size_t)rv * prows + jl] = ME_H ? wme * theirs : theirs;
      });
  if (far)
    far_pairs<NB_H>(L, ln, S.kl64, S, [&](int jl, int rv, int) {
      const RowState<BY_SITE, NB_H> st(S);
      const Site b = st.site(jl);
      double d[3];
      pair_vec(img, a, b, d);
      if (pair_inside<RULE>(d, a.s, b.s)) return;
      const double2 v = closed_dens<RULE>(d, a.s, b.s);
      rho += (NB_H ? st.occ(jl) : 1.0) * (NB_H ? v.y : v.x);
      share[(size_t)rv * prows + jl] = wme * (ME_H ? v.y : v.x);
    });
}

// Bound by the LDS (a row of 8 doubles) and the vector ALUs.  40^3 cells, events of
// a2c_fe_time_eval: 320 us, Gauss-Hermite rule 708 (278 and 621 with rows of
// degree 5, whose values were 1e-12 off at 1.1 A and 1e-13 beyond 5.0 A; 575 us
// with rows 8 doubles apart).
template <int RULE, int TBO, bool BY_SITE>
__global__ __launch_bounds__(TBO) __attribute__((amdgpu_waves_per_eu(4))) void k_dens_own64(
    const LatDev* __restrict__ lats, const int32_t* __restrict__ ob2l, int nblk, const double* __restrict__ gtab) {
  constexpr int ROWS = SNT * FP;
  __shared__ __align__(16) double tab[ROWS + EXPN];  // f_Pd, 2^(i/256)
  stage16(tab, gtab + S_FPD, ROWS / 2);
  stage16(tab + ROWS, gtab + S_EXP, EXPN / 2);
  __syncthreads();
  const int w = xcd_block() * (TBO / TB) + __builtin_amdgcn_readfirstlane(threadIdx.x / TB);
  if (w >= nblk) return;
  const LatDev& S = lats[ob2l[w]];
  if (S.rule != RULE) return;  // the other rule's instance serves this lattice
  const int K = S.kl64;
  const OwnerLane ln(S, w - S.owg0_64, K);
  if (ln.row >= ln.rows) return;  // whole lane groups
  const Image img = image_of(S);
  const int s = ln.pd ? ln.row : S.npd + ln.row;
  double wme;
  const Site a = own_site<BY_SITE>(S, ln, wme);
  double rho = 0.0;
  if (ln.pd) {
    dens_list<RULE, BY_SITE, false, false>(tab, tab + ROWS, S, ln, a, img, 1.0, rho);
    dens_list<RULE, BY_SITE, true, false>(tab, tab + ROWS, S, ln, a, img, 1.0, rho);
  } else {
    dens_list<RULE, BY_SITE, false, true>(tab, tab + ROWS, S, ln, a, img, wme, rho);
    dens_list<RULE, BY_SITE, true, true>(tab, tab + ROWS, S, ln, a, img, wme, rho);
  }
  rho = site_sum(rho, K);
  if (ln.ph == 0) gmem(S.epair)[s] = rho;  // free until the gradient pass
}

// by_site: rho, F' and the embedding energy in site order (a caller's density),
// else in row order (the passes that follow).
template <int DM>
__global__ __launch_bounds__(TB) void k_dens_recv64(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l,
                                                    int rq, double eps, int by_site) {
  const int v = xcd_block(), blk = v / rq;
  const LatDev& S = lats[b2l[blk]];
  const RecvLane ln(S, blk - S.blk0, v % rq);
  const int s = ln.s;
  if (ln.idle || s >= S.npd + S.nh) return;
  const double* __restrict__ xo = S.xrow;
  const bool pd = s < S.npd;
  const int row = pd ? s : s - S.npd;
  double rho = 0.0;
#pragma unroll
  for (int side = 0; side < 2; ++side) {  // shares arrive weighted by their senders
    const Ell& L = pd ? (side ? S.pdh : S.pdpd) : (side ? S.hh : S.hpd);
    row_shares<RECV_RU_SCALAR, double>(L, row, ln.ph, ln.G, [&](double v) { rho += v; });
  }
  rho = ln.sum(rho) + S.epair[s];
  if (ln.ph) return;
  rho *= S.rule == GH3 ? 1.0 : QW;
  const double xs = pd ? 1.0 : xo[row];
  const eam::VD F = pd ? eam::F_Pd_vd(rho) : eam::F_H_vd(rho);
  const int o = !by_site ? s : pd ? site_of_row(row, S.npd) : S.npd + site_of_row(row, S.nh);
  S.rho[o] = rho;
  S.Fp[o] = DM == A2C_DERIV_FD ? dF<DM>(pd, rho, eps) : F.d;
  S.emb[o] = xs * F.v;
}

// One node inside the tables: the pair energy phi and cu = SH dE/ds, E = F'_i f_j
// + F'_j f_i + phi.  FP multiplies f_Pd', FH f_H' / |r| (it carries FH_D).
constexpr int G_PH = S_PH - S_PD, G_EXP = S_EXP - S_PD;  // of the staged part
constexpr double FH_D = 0.5 * SH * FH_K * 11.0025;
template <int KIND, bool TAIL>
__device__ __forceinline__ void node_coef(const double* tab, const double* exptab, double x, double FP_, double FH,
                                          double& phi, double& cu) {
  const double* row = nullptr;
  SPos p{};
  if (KIND != 3) {
    p = s_pos(x);
    row = row_at<GP>(tab, p.k);
  }
  if (KIND == 0) {
    poly_vd<PHD>(row + 8, p.u, phi, cu);
    cu = fma(FP_, poly<GD>(row, p.u), cu);
  } else {
    double r, ri, fh, d;
    (void)fH_s<TAIL>(exptab, s_of(x), r, ri, fh);
    phi_r(tab + G_PH + (KIND == 3 ? 8 : 0), r, phi, d);
    cu = fma(FH, fh, (0.5 * SH * RINV) * d);
    cu = KIND == 3 ? cu * ri : fma(cu, ri, FP_ * poly<GD>(row, p.u));
  }
}

struct PairSums {
  double pe;        // sum of phi
  double g[3];      // q-gradient of this site (the partner's is -g)
  double gsi, gsj;  // sigma terms of both ends
};
// 12-point sums.  Site e's points are r = d +- a e_c with a = ai for the site
// and -aj for its partner.  With u = 2 SINV cu = (dE/dr) / |r| per node, T_c the
// difference of u between the two points of an axis, U_e their sum:
//   q-gradient  sum u r = d (U_i + U_j) + sum_e a T,
//   sigma terms d . T + a U (site i), its negative (partner).
// One axis of one site (2 nodes) per trip, the components rotating through d0
// and h2: more rows in flight would not fit the registers of 4 waves per SIMD.
template <int KIND, bool TAIL>
__device__ __forceinline__ PairSums pair_sums12(const double* tab, const double* exptab, const Nodes12& n,
                                                const double d[3], double ai, double aj, double FP, double FH) {
  double pe = 0.0, su = 0.0, d0 = d[0], d1 = d[1], d2 = d[2], h0 = 0.0, h1 = 0.0, h2 = 0.0;
  double a = ai, xb = n.xi, g = n.gi;
  PairSums p;
#pragma unroll 1
  for (int e = 0; e < 2; ++e) {
    double ue = 0.0, se = 0.0;
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
      const double t = g * d0;
      double phi0, phi1, u0, u1;
      node_coef<KIND, TAIL>(tab, exptab, xb + t, FP, FH, phi0, u0);
      node_coef<KIND, TAIL>(tab, exptab, xb - t, FP, FH, phi1, u1);
      pe += phi0 + phi1;
      const double T = u0 - u1;
      ue += u0 + u1;
      se = fma(d0, T, se);
      const double h = fma(a, T, h0), dt = d0;
      h0 = h1;
      h1 = h2;
      h2 = h;
      d0 = d1;
      d1 = d2;
      d2 = dt;
    }
    su += ue;
    p.gsj = -(2.0 * SINV) * fma(a, ue, se);
    if (e == 0) p.gsi = -p.gsj;
    a = -aj;
    xb = n.xj;
    g = -n.gj;
  }
  p.pe = pe;
  p.g[0] = (2.0 * SINV) * fma(d[0], su, h0);
  p.g[1] = (2.0 * SINV) * fma(d[1], su, h1);
  p.g[2] = (2.0 * SINV) * fma(d[2], su, h2);
  return p;
}
// Gauss-Hermite sums.  With u_k = w_k (dE/dr) / |r_k| and the node offsets a_k:
// U = sum u, V = sum u a, Wn = sum u |a|^2;
//   q-gradient  sum u r = d U + sqrt(3) s V,
//   Sz = sum u (r . z) = sqrt(3) d . V + 3 s Wn,  d/dsigma_k = Sz sigma_k / s.
// Weights 4 and 1 per axis, divided by 216 at the end; three nodes per trip.
template <int KIND, bool TAIL>
__device__ __forceinline__ PairSums pair_sums27(const double* tab, const double* exptab, const Nodes27& q,
                                                const double d[3], double sd, double si, double sj, double FP,
                                                double FH) {
  double pe = 0.0, U = 0.0, V0 = 0.0, V1 = 0.0, V2 = 0.0, Wn = 0.0;
#pragma unroll 1
  for (int a2 = -1; a2 <= 1; ++a2) {
#pragma unroll 1
    for (int a1 = -1; a1 <= 1; ++a1) {
      const double n2 = (double)(a2 * a2 + a1 * a1);
      const double xb = q.x0 + q.n1 * n2 + ((double)a2 * q.t[2] + (double)a1 * q.t[1]);
      const double w = (a2 ? 1.0 : 4.0) * (a1 ? 1.0 : 4.0);
      double f0, fm, fp, c0, cm, cp;
      node_coef<KIND, TAIL>(tab, exptab, xb, FP, FH, f0, c0);
      node_coef<KIND, TAIL>(tab, exptab, xb + q.n1 - q.t[0], FP, FH, fm, cm);
      node_coef<KIND, TAIL>(tab, exptab, xb + q.n1 + q.t[0], FP, FH, fp, cp);
      pe = fma(w, fma(4.0, f0, fm + fp), pe);
      const double e = cm + cp, u = w * fma(4.0, c0, e);
      U += u;
      V0 = fma(w, cp - cm, V0);
      V1 = fma((double)a1, u, V1);
      V2 = fma((double)a2, u, V2);
      Wn = fma(w, e, fma(n2, u, Wn));
    }
  }
  constexpr double Q = 2.0 * SINV / 216.0;
  const double sv = GH_Z * sd;
  PairSums p;
  p.pe = pe * (1.0 / 216.0);
  p.g[0] = Q * fma(d[0], U, sv * V0);
  p.g[1] = Q * fma(d[1], U, sv * V1);
  p.g[2] = Q * fma(d[2], U, sv * V2);
  const double sz = Q * fma(GH_Z, fma(d[0], V0, fma(d[1], V1, d[2] * V2)), 3.0 * sd * Wn);
  p.gsi = sz * (si / sd);
  p.gsj = sz * (sj / sd);
  return p;
}
// One pair in closed form, node by node.
template <int RULE, int KIND>
__device__ __forceinline__ PairSums closed_sums(const double d[3], double si, double sj, double Fi, double Fj) {
  const Closed<RULE> q(d, si, sj);
  PairSums p{};
  double sz = 0.0;
#pragma unroll 1
  for (int k = 0; k < Closed<RULE>::N; ++k) {
    double z[3], w, phi, c;
    const double r = q.node(k, z, w);
    pair_point<A2C_DERIV_ANALYTIC, KIND>(r, Fi, Fj, 0.0, phi, c);
    p.pe += w * phi;
    const double u = w * c / r;
    double ro = 0.0;  // r . z
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const double rx = d[x] + z[x];
      p.g[x] += u * rx;
      ro += rx * z[x];
    }
    if (RULE == GH3) sz += u * ro;
    else if (k < 6) p.gsi += u * ro / q.ai;
    else p.gsj += u * ro / q.aj;
  }
  if (RULE == GH3) {  // z = s (node): d/dsigma_k = (sum u r . node) sigma_k / s
    p.gsi = sz * si / (q.sd * q.sd);
    p.gsj = sz * sj / (q.sd * q.sd);
  }
  return p;
}
// false, and zeros, if a node lies outside the tables
template <int RULE, int KIND>
__device__ __forceinline__ bool pair_both(const double* tab, const double* exptab, const double d[3], double si,
                                          double sj, double Fi, double Fj, PairSums& p) {
  const double FP = KIND == 0 ? Fi + Fj : (KIND == 1 ? Fj : Fi);           // F' of the H site multiplies f_Pd'
  const double FH = FH_D * (KIND == 3 ? Fi + Fj : (KIND == 1 ? Fi : Fj));  // F' of the Pd site f_H'
  bool in;
  p = PairSums{};
  if (RULE == GH3) {
    const double sd = sqrt(fma(si, si, sj * sj));
    const Nodes27 n(d, sd);
    in = inside(n.lo, n.hi);
    if (in) {
      if (KIND != 0 && on_tail(n.hi)) p = pair_sums27<KIND, true>(tab, exptab, n, d, sd, si, sj, FP, FH);
      else p = pair_sums27<KIND, false>(tab, exptab, n, d, sd, si, sj, FP, FH);
    }
  } else {
    const double ai = SQ6 * si, aj = SQ6 * sj;
    const Nodes12 n(d, ai, aj);
    in = inside(n.lo, n.hi);
    if (in) {
      if (KIND != 0 && on_tail(n.hi)) p = pair_sums12<KIND, true>(tab, exptab, n, d, ai, aj, FP, FH);
      else p = pair_sums12<KIND, false>(tab, exptab, n, d, ai, aj, FP, FH);
    }
  }
  return in;
}

struct Own {
  double e = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0, gs = 0.0;
};
template <int RULE, int KIND>
__device__ __forceinline__ void grad_list(const double* tab, const double* exptab, const LatDev& S,
                                          const OwnerLane& ln, const Site& a, double Fi, const Image& img, double wme,
                                          Own& o) {
  constexpr bool ME_H = KIND >= 2, NB_H = KIND & 1;
  const Ell& L = ME_H ? (NB_H ? S.hh : S.hpd) : (NB_H ? S.pdh : S.pdpd);
  const Ell& P = ME_H ? (NB_H ? S.hh : S.pdh) : (NB_H ? S.hpd : S.pdpd);  // partner rows
  A2C_GLOBAL double4* __restrict__ share = gmem(reinterpret_cast<double4*>(P.rbuf));
  const size_t prows = P.rows;
  const A2C_GLOBAL double* Fp = gmem((const double*)S.Fp) + (NB_H ? S.npd : 0);
  bool far = false;
  owned_pairs<NB_H>(
      L, ln, S.kl64, S, [=](int j) { return Fp[j]; },
      [&](const Site& b) {
        Pair64 p;
        pair_vec(img, a, b, p.d);
        p.s = b.s;
        return p;
      },
      [&](const Pair64& q, double Fj, double wj, int jl, int rv) {
        PairSums p;
        far |= !pair_both<RULE, KIND>(tab, exptab, q.d, a.s, q.s, Fi, Fj, p);
        o.e += wj * p.pe;
        o.g0 += wj * p.g[0];
        o.g1 += wj * p.g[1];
        o.g2 += wj * p.g[2];
        o.gs += wj * p.gsi;
        // the partner's share leaves weighted by the sender's occupancy
        const double w = ME_H ? wme : 1.0;
        share[(size_t)rv * prows + jl] = make_double4(-w * p.g[0], -w * p.g[1], -w * p.g[2], w * p.gsj);
      });
  if (far)
    far_pairs<NB_H>(L, ln, S.kl64, S, [&](int jl, int rv, int j) {
      const Site b = load_row(gmem((const double2*)S.qxy), gmem((const double2*)S.qzs), j);
      double d[3];
      pair_vec(img, a, b, d);
      if (pair_inside<RULE>(d, a.s, b.s)) return;
      const PairSums p = closed_sums<RULE, KIND>(d, a.s, b.s, Fi, S.Fp[j]);
      const double wj = NB_H ? S.xrow[jl] : 1.0;
      o.e += wj * p.pe;
      o.g0 += wj * p.g[0];
      o.g1 += wj * p.g[1];
      o.g2 += wj * p.g[2];
      o.gs += wj * p.gsi;
      share[(size_t)rv * prows + jl] = make_double4(-wme * p.g[0], -wme * p.g[1], -wme * p.g[2], wme * p.gsj);
    });
}

// Bound by the LDS, with the vector ALUs close behind, at 2 waves per SIMD (the
// tables leave one workgroup per CU; 1024 lanes, 4 waves per SIMD, spill).  40^3
// cells, events of a2c_fe_time_eval: 670 us, Gauss-Hermite rule 1368 (562 and 1112
// with rows of degree 5, phi_HH in s and phi_Pd's last coefficients as floats;
// 1017 us with rows 17 doubles apart, read as 8-byte words).  Gradient error against
// 80-bit arithmetic (3^3 and 4^3 cells): 1e-14 to 3e-14; 3e-13 to 8e-13 with those
// rows, 4e-12 to 1e-11 with closed-form Pd slopes.
template <int RULE, int TBO>
__global__ __launch_bounds__(TBO) __attribute__((amdgpu_waves_per_eu(TBO / 256))) void k_grad_own64(
    const LatDev* __restrict__ lats, const int32_t* __restrict__ ob2l, int nblk, const double* __restrict__ gtab) {
  __shared__ __align__(16) double tab[G_EXP + EXPN];
  stage16(tab, gtab + S_PD, (G_EXP + EXPN) / 2);
  __syncthreads();
  const int w = xcd_block() * (TBO / TB) + __builtin_amdgcn_readfirstlane(threadIdx.x / TB);
  if (w >= nblk) return;
  const LatDev& S = lats[ob2l[w]];
  if (S.rule != RULE) return;  // the other rule's instance serves this lattice
  const int K = S.kl64;
  const OwnerLane ln(S, w - S.owg0_64, K);
  if (ln.row >= ln.rows) return;  // whole lane groups
  const double* exptab = tab + G_EXP;
  const Image img = image_of(S);
  const int s = ln.pd ? ln.row : S.npd + ln.row;
  const Site a = load_row(gmem((const double2*)S.qxy), gmem((const double2*)S.qzs), s);
  const double Fi = gmem((const double*)S.Fp)[s];
  Own o;
  if (ln.pd) {
    grad_list<RULE, 0>(tab, exptab, S, ln, a, Fi, img, 1.0, o);
    grad_list<RULE, 1>(tab, exptab, S, ln, a, Fi, img, 1.0, o);
  } else {
    const double wme = gmem((const double*)S.xrow)[ln.row];
    grad_list<RULE, 2>(tab, exptab, S, ln, a, Fi, img, wme, o);
    grad_list<RULE, 3>(tab, exptab, S, ln, a, Fi, img, wme, o);
  }
  o.e = site_sum(o.e, K);
  o.g0 = site_sum(o.g0, K);
  o.g1 = site_sum(o.g1, K);
  o.g2 = site_sum(o.g2, K);
  o.gs = site_sum(o.gs, K);
  if (ln.ph != 0) return;
  gmem(S.gown)[s] = make_double4(o.g0, o.g1, o.g2, o.gs);
  gmem(S.epair)[s] = o.e;
}

__global__ __launch_bounds__(TB) void k_grad_recv64(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l,
                                                 int rq) {
  const int v = xcd_block(), blk = v / rq;
  const LatDev& S = lats[b2l[blk]];
  const RecvLane ln(S, blk - S.blk0, v % rq);
  if (ln.idle) return;
  const int s = ln.s;
  double fs = 0.0, sl = 0.0;
  if (s < S.npd + S.nh) {
    const double* __restrict__ xo = S.xrow;
    const bool pd = s < S.npd;
    const int row = pd ? s : s - S.npd;
    double* __restrict__ G = S.G;
    const size_t site = pd ? site_of_row(row, S.npd) : S.npd + site_of_row(row, S.nh);
    double g0 = 0.0, g1 = 0.0, g2 = 0.0, gs = 0.0;
    if (ln.ph == 0) {
      const double4 own = S.gown[s];
      g0 = own.x; g1 = own.y; g2 = own.z; gs = own.w;
    }
#pragma unroll
    for (int side = 0; side < 2; ++side) {  // shares arrive weighted by their senders
      const Ell& L = pd ? (side ? S.pdh : S.pdpd) : (side ? S.hh : S.hpd);
      row_shares<RECV_RU_WIDE, double4>(L, row, ln.ph, ln.G, [&](const double4& v) {
        g0 += v.x; g1 += v.y; g2 += v.z;
        gs += v.w;
      });
    }
    g0 = ln.sum(g0); g1 = ln.sum(g1); g2 = ln.sum(g2); gs = ln.sum(gs);
    const double xi = pd ? 1.0 : xo[row];
    const double sg = S.qzs[s].y;
    const double T = S.T;
    const bool gh = S.rule == GH3;
    const double qw = gh ? 1.0 : QW, sq = gh ? 1.0 : SQ6;
    const double V = S.emb[s] + qw * xi * S.epair[s];  // owned pairs carry their full energy
    const double sc = qw * xi / T;
    if (ln.ph == 0) {
      g0 *= sc;
      g1 *= sc;
      g2 *= sc;
      gs = sq * sc * gs - 3.0 * KB * xi / sg;
      G[4 * site + 0] = g0;
      G[4 * site + 1] = g1;
      G[4 * site + 2] = g2;
      G[4 * site + 3] = gs;
      fs = V / T - 3.0 * KB * xi * log(sg);
      sl = site_slope(S, site, g0, g1, g2, gs);
    }
  }
  finish_objective(S, ln, fs, sl);
}

// ================================================================ chemical potential
// f_H and phi (phi_PdH, or phi_HH for an H neighbor) summed over a pair's nodes,
// with the rule's weights; false, and zeros, if a node lies outside the tables.
constexpr int C_EXP = S_EXP - S_PH;  // of the staged part
template <bool NB_H, bool TAIL>
__device__ __forceinline__ void node_fh_phi(const double* tab, const double* exptab, double x, double w, double& sf,
                                            double& sp) {
  double r, ri, sl;
  sf = fma(w, fH_s<TAIL>(exptab, s_of(x), r, ri, sl), sf);
  const double y = fma(r, RINV, RB);
  sp = fma(w, poly<RD>(row_at<RP>(tab + (NB_H ? 8 : 0), (int)y), eam::fract(y)), sp);
}
template <bool NB_H, bool TAIL>
__device__ __forceinline__ void fh_phi_sums27(const double* tab, const double* exptab, const Nodes27& q, double& sf,
                                              double& sp) {
#pragma unroll 1
  for (int k = 0; k < 9; ++k) {
    const int a2 = k / 3 - 1, a1 = k % 3 - 1;
    const double xb = q.x0 + q.n1 * (double)(a2 * a2 + a1 * a1) + ((double)a2 * q.t[2] + (double)a1 * q.t[1]);
    const double w = (a2 ? 1.0 : 4.0) * (a1 ? 1.0 : 4.0);
#pragma unroll
    for (int a0 = -1; a0 <= 1; ++a0)
      node_fh_phi<NB_H, TAIL>(tab, exptab, a0 ? xb + q.n1 + a0 * q.t[0] : xb, a0 ? w : 4.0 * w, sf, sp);
  }
  sf *= 11.0025 / 216.0;
  sp *= 1.0 / 216.0;
}
template <bool NB_H, bool TAIL>
__device__ __forceinline__ void fh_phi_sums12(const double* tab, const double* exptab, const Nodes12& q,
                                              const double d[3], double& sf, double& sp) {
  double d0 = d[0], d1 = d[1], d2 = d[2];
#pragma unroll 1
  for (int c = 0; c < 3; ++c) {
    const double ti = q.gi * d0, tj = q.gj * d0;
    const double x[4] = {q.xi + ti, q.xi - ti, q.xj - tj, q.xj + tj};
#pragma unroll
    for (int k = 0; k < 4; ++k) node_fh_phi<NB_H, TAIL>(tab, exptab, x[k], 1.0, sf, sp);
    d0 = d1;
    d1 = d2;
  }
  sf *= 11.0025 * QW;
  sp *= QW;
}
template <int RULE, bool NB_H>
__device__ __forceinline__ bool pair_fh_phi(const double* tab, const double* exptab, const double d[3], double si,
                                            double sj, double& sf, double& sp) {
  sf = sp = 0.0;
  if (RULE == GH3) {
    const Nodes27 q(d, sqrt(fma(si, si, sj * sj)));
    if (!inside(q.lo, q.hi)) return false;
    if (on_tail(q.hi)) fh_phi_sums27<NB_H, true>(tab, exptab, q, sf, sp);
    else fh_phi_sums27<NB_H, false>(tab, exptab, q, sf, sp);
  } else {
    const Nodes12 q(d, SQ6 * si, SQ6 * sj);
    if (!inside(q.lo, q.hi)) return false;
    if (on_tail(q.hi)) fh_phi_sums12<NB_H, true>(tab, exptab, q, d, sf, sp);
    else fh_phi_sums12<NB_H, false>(tab, exptab, q, d, sf, sp);
  }
  return true;
}
template <int RULE, bool NB_H>
__device__ __forceinline__ void closed_fh_phi(const double d[3], double si, double sj, double& sf, double& sp) {
  const Closed<RULE> q(d, si, sj);
  sf = sp = 0.0;
#pragma unroll 1
  for (int k = 0; k < Closed<RULE>::N; ++k) {
    double z[3], w;
    const double r = q.node(k, z, w);
    sf += w * eam::f_H(r);
    sp += w * eam::phi_morse<NB_H>(r);
  }
  sf *= rule_qw<RULE>();
  sp *= rule_qw<RULE>();
}

// The listed neighbors of H row `row` (full list L, site order), K lanes to a
// row: sum += w_j (F'_j f_H + phi + corr_j), xs += w_j.  A pair's state is loaded a
// pair ahead.
template <int RULE, bool NB_H>
__device__ __forceinline__ void chem_list(const double* tab, const double* exptab, const LatDev& S, const Ell& L,
                                          const A2C_GLOBAL double* corr, int row, int ph, int K, const Site& a,
                                          const Image& img, double& sum, double& xs) {
  const A2C_GLOBAL double2* __restrict__ qxy = gmem((const double2*)S.qxy) + (NB_H ? S.npd : 0);
  const A2C_GLOBAL double2* __restrict__ qzs = gmem((const double2*)S.qzs) + (NB_H ? S.npd : 0);
  const A2C_GLOBAL double* __restrict__ Fp = gmem((const double*)S.Fp) + (NB_H ? S.npd : 0);
  const A2C_GLOBAL double* __restrict__ w = gmem((const double*)S.xrow);
  const int site = site_of_row(row, S.nh), jrows = NB_H ? S.nh : S.npd;
  const A2C_GLOBAL int32_t* __restrict__ idx = gmem((const int32_t*)L.idx) + site;
  const size_t rows = L.rows;
  const int n = gmem((const int32_t*)L.cnt)[site];
  corr += NB_H ? S.npd : 0;
  if (ph >= n) return;
  auto at = [&](int t) { return row_of_site(idx[(size_t)(t < n ? t : ph) * rows], jrows); };
  int j = at(ph), jn = at(ph + K);
  Site b = load_row(qxy, qzs, j);
  double Fj = Fp[j], cj = corr[j], wj = NB_H ? w[j] : 1.0;
  bool far = false;
  for (int t = ph; t < n; t += K) {
    Pair64 p;
    pair_vec(img, a, b, p.d);
    p.s = b.s;
    const double Fc = Fj, cc = cj, wc = wj;
    b = load_row(qxy, qzs, jn);
    Fj = Fp[jn];
    cj = corr[jn];
    if (NB_H) wj = w[jn];
    jn = at(t + 2 * K);
    double sf, sp;
    const bool in = pair_fh_phi<RULE, NB_H>(tab, exptab, p.d, a.s, p.s, sf, sp);
    far |= !in;
    const double v = fma(Fc, sf, sp) + cc;
    xs += wc;
    if (in) sum += NB_H ? wc * v : v;
  }
  if (!far) return;
  for (int t = ph; t < n; t += K) {
    j = at(t);
    b = load_row(qxy, qzs, j);
    double d[3], sf, sp;
    pair_vec(img, a, b, d);
    if (pair_inside<RULE>(d, a.s, b.s)) continue;
    closed_fh_phi<RULE, NB_H>(d, a.s, b.s, sf, sp);
    sum += (NB_H ? w[j] : 1.0) * (fma(Fp[j], sf, sp) + corr[j]);
  }
}

// Chemical potential of the H sites (occupancy.hip has the formula), K lanes per
// row over the full lists, from rho and F' in row order.  24^3 cells: one lane per
// site and closed forms 353 us, this 118 us (4 waves per SIMD; LDS and FP64 units both
// busy); error against 80-bit arithmetic 1.3e-12 to 2.3e-12 before, 2.3e-15 to 4.3e-15
// now.
template <int RULE, int TBO>
__global__ __launch_bounds__(TBO) __attribute__((amdgpu_waves_per_eu(TBO / 256, TBO / 256))) void k_chem64(const LatDev* __restrict__ lat, int units, int K,
                                                const double* __restrict__ gtab, ChemArgs c) {
  __shared__ __align__(16) double tab[C_EXP + EXPN];
  stage16(tab, gtab + S_PH, (C_EXP + EXPN) / 2);  // phi_PdH, phi_HH, 2^(i/256)
  __syncthreads();
  const double* exptab = tab + C_EXP;
  const int u = xcd_block() * (TBO / TB) + __builtin_amdgcn_readfirstlane(threadIdx.x / TB);
  if (u >= units) return;
  const LatDev& S = *lat;
  const int lane = (int)threadIdx.x % TB, sh = 31 - __builtin_clz(K);
  const int row = u * (TB >> sh) + (lane >> sh), ph = lane & (K - 1);
  if (row >= S.nh) return;  // whole lane groups
  const int site = site_of_row(row, S.nh);
  if (c.full[site] == 1) return;  // fully occupied reservoir: gamma untouched
  const int s = S.npd + row;
  const Image img = image_of(S);
  const Site a = load_row(gmem((const double2*)S.qxy), gmem((const double2*)S.qzs), s);
  const A2C_GLOBAL double* corr = gmem(c.corr);
  double sum = 0.0, nP = 0.0, Xa = 0.0;
  chem_list<RULE, false>(tab, exptab, S, S.hpd, corr, row, ph, K, a, img, sum, nP);
  chem_list<RULE, true>(tab, exptab, S, S.hh, corr, row, ph, K, a, img, sum, Xa);
  sum = site_sum(sum, K);
  Xa = site_sum(Xa, K);
  nP = site_sum(nP, K);
  if (ph != 0) return;
  const double T = S.T, x = S.xrow[row];
  sum += eam::F_H(S.rho[s]);
  sum += 0.5 * T * c.ch[0] * (c.ch[1] * nP * nP + 2.0 * c.ch[2] * nP * Xa + c.ch[3] * Xa * Xa);
  const double raw = (x > 0.0 && x < 1.0) ? log(x / (1.0 - x)) + sum / (KB * T) : 0.0;
  double g = raw + 1.5;
  if (g > c.gamma_bd) {
    g = c.gamma_bd;
    if (x > 0.9999) c.full[site] = 1;
  }
  c.gamma[site] = g;
}

// Row-order copies of the state and the occupancy for the pair passes.
__global__ __launch_bounds__(TB) void k_rows(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l) {
  const int blk = xcd_block();
  const LatDev& S = lats[b2l[blk]];
  const int s = (blk - S.blk0) * TB + threadIdx.x;
  copy_row(S, s);
}

}  // namespace

// One block per lattice: fixed-order sum of its block partials.
__global__ __launch_bounds__(1024) void k_final_sum(const LatDev* __restrict__ lats) {
  __shared__ double red[1024];
  const LatDev& S = lats[blockIdx.x];
  const int n = site_blocks(S.npd + S.nh);
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) acc += S.part[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *S.f = red[0];
}

namespace {
// Launch the instance of each quadrature rule present in the launch.
template <template <int> class K, class... A>
int per_rule(const Launch& L, int nblk, A... args) {
  if (nblk == 0) return A2C_OK;
  if (L.rules & (1 << A2C_QUAD_R12))
    hipLaunchKernelGGL(K<A2C_QUAD_R12>::fn, dim3(nblk), dim3(TB), 0, L.stream, args...);
  if (L.rules & (1 << GH3)) hipLaunchKernelGGL(K<GH3>::fn, dim3(nblk), dim3(TB), 0, L.stream, args...);
  return hipGetLastError() == hipSuccess ? A2C_OK : A2C_EHIP;
}
template <int R> struct DensFd { static constexpr auto fn = k_density64<A2C_DERIV_FD, R>; };
template <int R> struct DensAn { static constexpr auto fn = k_density64<A2C_DERIV_ANALYTIC, R>; };
template <int R> struct GradFd { static constexpr auto fn = k_grad64<A2C_DERIV_FD, R>; };
template <int R> struct GradAn { static constexpr auto fn = k_grad64<A2C_DERIV_ANALYTIC, R>; };
// Owner launches: workgroups of TBO lanes, TBO / 256 units each.
template <template <int, int> class K, int TBO>
int owners(const Launch& L) {
  if (L.onblk == 0) return A2C_OK;
  const dim3 grid((L.onblk + TBO / TB - 1) / (TBO / TB));
  if (L.rules & (1 << A2C_QUAD_R12))
    hipLaunchKernelGGL((K<A2C_QUAD_R12, TBO>::fn), grid, dim3(TBO), 0, L.stream, L.lats, L.ob2l, L.onblk, L.tab64);
  if (L.rules & (1 << GH3))
    hipLaunchKernelGGL((K<GH3, TBO>::fn), grid, dim3(TBO), 0, L.stream, L.lats, L.ob2l, L.onblk, L.tab64);
  return hipGetLastError() == hipSuccess ? A2C_OK : A2C_EHIP;
}
// Up to a unit per CU (gradient pass, one workgroup per CU) or two (density
// pass) the units go to workgroups of their own; beyond, two to a workgroup, so
// that a CU holds 8 waves on one copy of the tables.
constexpr int GRAD_WIDE_UNITS = 256, DENS_WIDE_UNITS = 512;
template <int R, int T> struct DensOwn { static constexpr auto fn = k_dens_own64<R, T, false>; };
template <int R, int T> struct DensOwnFold { static constexpr auto fn = k_dens_own64<R, T, true>; };
// the row-order copies and the density pass
int run_dens_own(const Launch& L, Timing* tm) {
  const bool fold = fold_rows(L), wide = L.onblk > DENS_WIDE_UNITS;
  if (!fold) {
    if (tm) tm->mark(L.stream, "rows");
    if (run_rows(L)) return A2C_EHIP;
  }
  if (tm) tm->mark(L.stream, "dens_own64");
  if (fold) return wide ? owners<DensOwnFold, 512>(L) : owners<DensOwnFold, 256>(L);
  return wide ? owners<DensOwn, 512>(L) : owners<DensOwn, 256>(L);
}
template <int R, int T> struct GradOwn { static constexpr auto fn = k_grad_own64<R, T>; };
}  // namespace

// rho, F', embedding energy from full lists, in site order
static int run_density64(const Launch& L) {
  if (L.deriv_mode == A2C_DERIV_FD) return per_rule<DensFd>(L, L.nblk, L.lats, L.b2l, L.fd_eps);
  return per_rule<DensAn>(L, L.nblk, L.lats, L.b2l, L.fd_eps);
}

int run_eval64(const Launch& L, Timing* tm) {
  if (L.deriv_mode == A2C_DERIV_ANALYTIC && !L.full_pairs64) {
    if (L.nblk > 0) {
      if (run_dens_own(L, tm)) return A2C_EHIP;
      if (tm) tm->mark(L.stream, "dens_recv64");
      hipLaunchKernelGGL(k_dens_recv64<A2C_DERIV_ANALYTIC>, dim3(L.nblk * L.rq), dim3(TB), 0, L.stream, L.lats, L.b2l,
                         L.rq, 0.0, 0);
      if (hipGetLastError() != hipSuccess) return A2C_EHIP;
      if (tm) tm->mark(L.stream, "grad_own64");
      if (L.onblk > GRAD_WIDE_UNITS ? owners<GradOwn, 512>(L) : owners<GradOwn, 256>(L)) return A2C_EHIP;
      if (tm) tm->mark(L.stream, "grad_recv64");
      hipLaunchKernelGGL(k_grad_recv64, dim3(L.nblk * L.rq), dim3(TB), 0, L.stream, L.lats, L.b2l, L.rq);
      if (hipGetLastError() != hipSuccess) return A2C_EHIP;
    }
    if (tm) tm->mark(L.stream, nullptr);
    return A2C_OK;
  }
  if (tm) tm->mark(L.stream, "density64");
  if (int rc = run_density64(L)) return rc;
  if (tm) tm->mark(L.stream, "grad64");
  if (L.deriv_mode == A2C_DERIV_FD) {
    if (per_rule<GradFd>(L, L.nblk, L.lats, L.b2l, L.fd_eps)) return A2C_EHIP;
  } else if (per_rule<GradAn>(L, L.nblk, L.lats, L.b2l, L.fd_eps)) {
    return A2C_EHIP;
  }
  if (tm) tm->mark(L.stream, "final_sum");
  if (int rc = run_final_sum(L)) return rc;
  if (tm) tm->mark(L.stream, nullptr);
  return A2C_OK;
}

bool fold_rows(const Launch& L) { return L.nblk <= FOLD_BLOCKS && !L.empty; }
int run_rows(const Launch& L) {
  hipLaunchKernelGGL(k_rows, dim3(L.nblk), dim3(TB), 0, L.stream, L.lats, L.b2l);
  return hipGetLastError() == hipSuccess ? A2C_OK : A2C_EHIP;
}

int run_final_sum(const Launch& L) {
  if (L.nlat == 0) return A2C_OK;
  hipLaunchKernelGGL(k_final_sum, dim3(L.nlat), dim3(1024), 0, L.stream, L.lats);
  return hipGetLastError() == hipSuccess ? A2C_OK : A2C_EHIP;
}

// The tables of the owner passes (see "pair-once"), from the closed forms in
// long double.
void host_tables64_s(std::vector<double>& t) {
  static const std::vector<double> built = [] {
    using LD = long double;
    std::vector<double> out((size_t)S_SIZE, 0.0);
    const LD PI = 3.14159265358979323846264338327950288L, h = 1 / (LD)SINV, s0 = -(LD)SB / SINV;
    auto node = [&](int i, int n) { return 0.5L - 0.5L * cosl((2 * i + 1) * PI / (2.0L * n)); };
    constexpr int MAXC = 12;
    // polynomial through (u[i], y[i]), i < n, as monomials
    auto through = [](const LD* u, const LD* y, int n, LD* m) {
      LD c[MAXC];
      for (int i = 0; i < n; ++i) c[i] = y[i];
      for (int j = 1; j < n; ++j)
        for (int i = n - 1; i >= j; --i) c[i] = (c[i] - c[i - 1]) / (u[i] - u[i - j]);
      for (int q = 0; q < MAXC; ++q) m[q] = 0;
      for (int i = n - 1; i >= 0; --i) {
        for (int q = MAXC - 1; q > 0; --q) m[q] = m[q - 1] - u[i] * m[q];
        m[0] = c[i] - u[i] * m[0];
      }
    };
    enum { VALUE, SLOPE, BOTH };
    // rows of degree deg at out[base + k pitch]; g: value and slope in r
    auto fill = [&](int base, int pitch, int rows, bool in_r, int deg, int fit, auto g) {
      for (int k = 0; k < rows; ++k) {
        auto at = [&](LD u) {
          const LD r = in_r ? (k + u - RB) / RINV : sqrtl(s0 + (k + u) * h);
          const eam::VDT<LD> v = g(r);
          return eam::VDT<LD>{v.v, v.d * (in_r ? 1 / (LD)RINV : h / (2 * r))};  // d/du
        };
        const int n = fit == BOTH ? deg : deg + 1;
        LD u[MAXC], y[MAXC], m[MAXC];
        for (int i = 0; i < n; ++i) {
          u[i] = node(i, n);
          y[i] = fit == VALUE ? at(u[i]).v : at(u[i]).d;
        }
        through(u, y, n, m);
        if (fit == BOTH) {  // the slope's integral, with the value's mean over the Chebyshev points
          for (int q = deg; q > 0; --q) m[q] = m[q - 1] / q;
          m[0] = 0;
          LD c = 0;
          for (int i = 0; i < 8; ++i) {
            const LD w = node(i, 8);
            LD v = 0;
            for (int q = deg; q >= 0; --q) v = v * w + m[q];
            c += at(w).v - v;
          }
          m[0] = c / 8;
        }
        for (int q = 0; q <= deg; ++q) out[(size_t)base + (size_t)k * pitch + q] = (double)m[q];
      }
    };
    fill(S_FPD, FP, SNT, false, FD, VALUE, [](LD r) { return eam::f_Pd_vd<LD>(r); });
    fill(S_PD, GP, SNT, false, GD, SLOPE, [](LD r) { return eam::f_Pd_vd<LD>(r); });
    fill(S_PD + 8, GP, SNT, false, PHD, BOTH, [](LD r) { return eam::phi_Pd_vd<LD>(r, eam::f_Pd_vd<LD>(r)); });
    fill(S_PH, RP, RNT, true, RD, BOTH, [](LD r) { return eam::phi_morse_vd<0, LD>(r); });
    fill(S_PH + 8, RP, RNT, true, RD, BOTH, [](LD r) { return eam::phi_morse_vd<1, LD>(r); });
    for (int i = 0; i < EXPN; ++i) out[S_EXP + i] = (double)exp2l((LD)i / EXPN);
    return out;
  }();
  t = built;
}

// One EAM function (order of a2c_eam_tables) at r in [1, 6) as the passes take it
// from the tables t: value, and slope in r.
void pass_eval64(const std::vector<double>& t, int fn, double r, double& v, double& d) {
  const double s = r * r, x = fma(s, SINV, SB), *exptab = &t[S_EXP];
  const SPos p = s_pos(x);
  double r1, ri, sl;
  const double fh = fH_s<true>(exptab, s, r1, ri, sl);
  if (fn == 1) {
    v = 11.0025 * fh;
    d = FH_K * 11.0025 * sl;
  } else if (fn > 2) {
    phi_r(&t[S_PH + (fn == 3 ? 0 : 8)], r1, v, d);
    d *= RINV;
  } else {
    const double* row = row_at<GP>(&t[S_PD], p.k);
    if (fn == 0) {
      v = poly<FD>(row_at<FP>(&t[S_FPD], p.k), p.u);
      d = poly<GD>(row, p.u);
    } else {
      poly_vd<PHD>(row + 8, p.u, v, d);
    }
    d *= 2.0 * SINV * r;
  }
}

// FP64 tables in r (exported, a2c_eam_tables64): on each 0.05 A interval the polynomial (degree 8 for the
// exponential functions, 11 for the Pd polynomials) interpolating the
// long-double closed form at the Chebyshev points, in Newton form, expanded
// to monomials in u (all in long double); the switch radii 5.0, 5.05 and
// 5.35 A are interval boundaries.
void host_tables64(std::vector<double>& t) {
  static const std::vector<double> built = [] {
    using LD = long double;
    std::vector<double> out((size_t)T64_SIZE, 0.0);
    auto fill = [&](auto deg, size_t base, int pitch, auto g) {
      constexpr int D = decltype(deg)::value;
      const LD H = 0.05L, PI = 3.14159265358979323846264338327950288L;
      for (int k = 0; k < T64_N; ++k) {
        const LD a = 1.0L + H * k;
        LD u[D + 1], c[D + 1], m[D + 1] = {};
        for (int i = 0; i <= D; ++i) {
          u[i] = 0.5L - 0.5L * cosl((2 * i + 1) * PI / (2.0L * (D + 1)));
          c[i] = g(a + u[i] * H);
        }
        for (int j = 1; j <= D; ++j)  // divided differences
          for (int i = D; i >= j; --i) c[i] = (c[i] - c[i - 1]) / (u[i] - u[i - j]);
        for (int i = D; i >= 0; --i) {  // m <- m (u - u_i) + c_i
          LD n[D + 1] = {};
          for (int q = 0; q < D; ++q) {
            n[q + 1] += m[q];
            n[q] -= m[q] * u[i];
          }
          n[0] += c[i];
          for (int q = 0; q <= D; ++q) m[q] = n[q];
        }
        for (int q = 0; q <= D; ++q) out[base + (size_t)k * pitch + q] = (double)m[q];
      }
    };
    using D8 = std::integral_constant<int, T64_D>;
    using D11 = std::integral_constant<int, T64Q_D>;
    fill(D8{}, (size_t)T64_FH * T64_N * T64_P, T64_P, [](LD r) { return eam::f_H<LD>(r); });
    fill(D8{}, (size_t)T64_PHPDH * T64_N * T64_P, T64_P, [](LD r) { return eam::phi_morse<0, LD>(r); });
    fill(D8{}, (size_t)T64_PHH * T64_N * T64_P, T64_P, [](LD r) { return eam::phi_morse<1, LD>(r); });
    fill(D11{}, T64_PART1 + (size_t)T64Q_FPD * T64_N * T64Q_P, T64Q_P, [](LD r) { return eam::f_Pd<LD>(r); });
    fill(D11{}, T64_PART1 + (size_t)T64Q_PHPD * T64_N * T64Q_P, T64Q_P, [](LD r) { return eam::phi_Pd<LD>(r); });
    return out;
  }();
  t = built;
}

bool mixed_full_pairs() {
  static const bool full = [] {
    const char* v = getenv("A2C_MIXED_PAIRS");
    return v && std::string(v) == "full";
  }();
  return full;
}
bool fp64_full_pairs() {
  static const bool full = [] {
    const char* v = getenv("A2C_FP64_PAIRS");
    return v && std::string(v) == "full";
  }();
  return full;
}

static Launch single_launch(a2c_fe_ctx* c, bool fp64) {
  Launch L;
  L.mixed_full = mixed_full_pairs();
  L.full_pairs64 = fp64_full_pairs();
  L.lats = c->dlat;
  L.b2l = c->db2l;
  L.ob2l = c->db2l;
  L.onblk = owner_units(c->desc.n_pd, c->desc.n_h, lanes_per_site(c->N, fp64));
  L.nblk = lattice_blocks(c->N);
  L.rq = recv_lanes(c->N);
  L.empty = c->N == 0;
  L.nlat = 1;
  L.rules = 1 << c->desc.quad_rule;
  L.stream = c->stream;
  L.deriv_mode = c->desc.deriv_mode;
  L.fd_eps = c->desc.fd_eps;
  L.tab = c->dtab;
  L.tab64 = c->dtab64;
  return L;
}

// Density, F' and embedding energy of the context's lattice from the pair-once
// passes, in site or in row order.
int launch_density64(a2c_fe_ctx* c, const double* dX, bool by_site) {
  if (c->gen_on) return launch_density_gen(c, dX);
  if (int rc = sync_lattice(c, dX, c->dG, c->dF)) return rc;
  const Launch L = single_launch(c, true);
  if (run_dens_own(L, nullptr))
    return set_err(c, A2C_EHIP, "density64 launch failed");
  hipLaunchKernelGGL(L.deriv_mode == A2C_DERIV_FD ? k_dens_recv64<A2C_DERIV_FD> : k_dens_recv64<A2C_DERIV_ANALYTIC>,
                     dim3(L.nblk * L.rq), dim3(TB), 0, L.stream, L.lats, L.b2l, L.rq, L.fd_eps, (int)by_site);
  A2C_HIP(c, hipGetLastError());
  return A2C_OK;
}

// The chemical potential from what launch_density64 left in row order.  Up to a
// unit of 256 lanes per CU the units go to workgroups of their own; beyond, two
// or four share one, so that a CU's one copy of the tables serves all its waves.
template <int RULE>
static void launch_chem64_rule(a2c_fe_ctx* c, const ChemArgs& a) {
  // lanes per row as in the mixed passes: one species' full lists are a smaller, longer launch than the FP64 passes'
  const int K = lanes_per_site(c->N, false), units = owner_units(c->desc.n_h, K);
  auto go = [&](auto kernel, int tbo) {
    hipLaunchKernelGGL(kernel, dim3((units + tbo / TB - 1) / (tbo / TB)), dim3(tbo), 0, c->stream,
                       (const LatDev*)c->dlat, units, K, (const double*)c->dtab64, a);
  };
  if (units <= 256) go(k_chem64<RULE, 256>, 256);
  else if (units <= 512) go(k_chem64<RULE, 512>, 512);
  else go(k_chem64<RULE, 1024>, 1024);
}
int launch_chem64(a2c_fe_ctx* c, const ChemArgs& a) {
  if (c->desc.n_h <= 0) return A2C_OK;
  if (c->desc.quad_rule == A2C_QUAD_GH3) launch_chem64_rule<GH3>(c, a);
  else launch_chem64_rule<A2C_QUAD_R12>(c, a);
  A2C_HIP(c, hipGetLastError());
  return A2C_OK;
}

int launch_eval64(a2c_fe_ctx* c, const double* dX, double* dG, double* dF, bool timed, Timing* tm) {
  if (int rc = sync_lattice(c, dX, dG, dF)) return rc;
  if (run_eval64(single_launch(c, true), timed ? tm : nullptr)) return set_err(c, A2C_EHIP, "eval64 launch failed");
  return A2C_OK;
}

int launch_eval32(a2c_fe_ctx* c, const double* dX, double* dG, double* dF, bool timed, Timing* tm) {
  if (!c->dtab) return set_err(c, A2C_ESTATE, "tables not built");
  if (int rc = sync_lattice(c, dX, dG, dF)) return rc;
  if (run_eval32(single_launch(c, false), timed ? tm : nullptr)) return set_err(c, A2C_EHIP, "eval32 launch failed");
  return A2C_OK;
}

// Refresh the device descriptor of the context's lattice when the state,
// gradient or objective buffers (or the neighbor lists) changed.
int sync_lattice(a2c_fe_ctx* c, const double* dX, double* dG, double* dF) {
  if (!c->hlat) {  // pinned, at the first single-lattice launch (a batch's lattices never need it)
    A2C_HIP(c, hmalloc(&c->hlat, sizeof(LatDev)));
    new (c->hlat) LatDev();
    c->lat_dirty = true;
  }
  if (!c->db2l) {  // all-zero block -> lattice map: site blocks, or owner units at any lanes per site
    const size_t n = 4 * (size_t)(owner_units(c->N, MAX_LANES_PER_SITE) + 1);
    const DeviceScope on(c->desc.device);
    A2C_HIP(c, on.status());
    A2C_HIP(c, dmalloc(&c->db2l, n));
    A2C_HIP(c, hipMemsetAsync(c->db2l, 0, n, c->stream));
  }
  LatDev& h = *c->hlat;
  const int kl32 = lanes_per_site(c->N, false), kl64 = lanes_per_site(c->N, true);
  if (!c->lat_dirty && h.X == dX && h.G == dG && h.f == dF && h.kl32 == kl32 && h.kl64 == kl64) return A2C_OK;
  A2C_HIP(c, hipStreamSynchronize(c->stream));  // the pinned copy may still be in flight
  h = c->sys();
  h.blk0 = 0;
  h.kl32 = kl32;  // the launch grid (single_launch) takes K from the same table
  h.kl64 = kl64;
  h.owg0_32 = h.owg0_64 = 0;
  h.X = dX;
  h.G = dG;
  h.f = dF;
  A2C_HIP(c, hipMemcpyAsync(c->dlat, c->hlat, sizeof(LatDev), hipMemcpyHostToDevice, c->stream));
  c->lat_dirty = false;
  return A2C_OK;
}

}  // namespace a2c

// Host-only: the FP64 tables in r (layout in a2c_fe.h).
extern "C" int a2c_eam_tables64(double* out, int32_t cap) {
  std::vector<double> t;
  a2c::host_tables64(t);
  const int n = (int)t.size();
  if (out && cap >= n) std::memcpy(out, t.data(), sizeof(double) * n);
  return n;
}

// Host-only: an EAM function as the pair-once passes evaluate it (a2c_fe.h).
extern "C" int a2c_eam_pass(int32_t precision, int32_t fn, int32_t n, const double* r, double* r_at, double* v,
                            double* d) {
  if ((precision != A2C_PREC_FP64 && precision != A2C_PREC_MIXED) || fn < 0 || fn > 4 || n < 0) return A2C_EINVAL;
  if (n > 0 && (!r || !r_at || !v || !d)) return A2C_EINVAL;
  std::vector<double> t64;
  std::vector<float4> t32;
  if (precision == A2C_PREC_FP64) a2c::host_tables64_s(t64);
  else a2c::host_tables(t32), a2c::host_tables_s(t32);
  for (int i = 0; i < n; ++i) {
    if (!(r[i] >= 1.0 && r[i] < 5.999)) return A2C_EINVAL;
    if (precision == A2C_PREC_FP64) {
      r_at[i] = r[i];
      a2c::pass_eval64(t64, fn, r[i], v[i], d[i]);
    } else {
      r_at[i] = a2c::pass_eval32(t32, fn, r[i], v[i], d[i]);
    }
  }
  return A2C_OK;
}
