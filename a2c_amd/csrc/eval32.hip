// Mixed-precision objective + gradient (Minimizer::formFunctionAndGradient,
// minimizer.cpp:83-369): FP32 bulk quadrature, FP64 everywhere the error
// would not average out.
//
//   FP64: positions, the pair vector d = q_i - q_j (then rounded to FP32, so
//         the rounding is relative to |d| <= rc, not to the box size),
//         per-site accumulation of the per-pair sums, rho, F(rho), F'(rho),
//         the per-site objective share and the global reduction.
//   FP32: the 12 quadrature points of a pair: |r|^2 = |d|^2 + a^2 +- 2 a d_c
//         (each point displaces d along one axis by a = sqrt(6) sigma), and the
//         EAM functions there.  Under the Gauss-Hermite rule the 27 nodes
//         r_k = d + s sqrt(3) a_k (a_k in {-1,0,1}^3) have
//         |r_k|^2 = |d|^2 + 3 s^2 |a_k|^2 + 2 sqrt(3) s (a_k . d).
//
// The EAM functions are piecewise cubics built on the host in 80-bit long
// double, stored as FP32 coefficients in the local coordinate u in [0, 1) and
// staged in LDS.  The pair-once passes take them on a uniform grid in |r|^2
// (see "pair-once"), the full-list passes on one in |r|: cubic Hermite pieces
// of h = 0.01 A over [1, 6] A, switch radii 5.0, 5.05, 5.35 on grid nodes, 1/|r|
// by v_rsq_f32.  Beyond 6 A every function is the exponential tail of
// potential.cpp, evaluated directly.
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "eam64.hpp"
#include "fe_internal.hpp"
#include "pair_rows.hpp"

namespace a2c {
namespace {

constexpr int TB = SITE_BLOCK;
constexpr int NT = 500;               // intervals per table (h = 0.0125 would fit 32 KB of LDS, but the
                                      // f_Pd derivative error then reaches 1.4e-5 of its maximum)
constexpr float R0 = 1.0f, R1 = 6.0f, INVH = 100.0f;
constexpr double H64 = 0.01;
constexpr double QW = 1.0 / 12.0;     // 0.5/dim, quadrature.cpp:39
constexpr double SQ6 = 2.449489742783178098;
constexpr float SQ6F = 2.449489742783178098f;
constexpr int GH3 = A2C_QUAD_GH3;
constexpr float GHZF = 1.7320508075688772935f;  // Gauss-Hermite node sqrt(3)
// Gauss-Hermite weights times 6 per axis: 4, 1 and their products are exact in
// FP32, where 2/3 and 1/6 are not and leave the sum of the 27 weights 1e-7 off
// one (a bias of every density and pair energy); the receive passes divide by 216.
__device__ constexpr float ghwf(int a) { return a == 0 ? 4.0f : 1.0f; }
constexpr double GHQW = 1.0 / 216.0;
enum { T_FPD = 0, T_FH = 1, T_PHPD = 2, T_PHPDH = 3, T_PHH = 4, NTAB = 5 };

// Exponential tails beyond the switch radii: funRc * exp(k (r - rs)).
__constant__ float TAIL[NTAB][3] = {
    {0.001510569378297f, (float)(-0.077976566126292 / 0.001510569378297), 5.0f},
    {0.009986990526578f, (float)(-0.013075667086408 / 0.009986990526578), 5.35f},
    {-0.016958780164980f, (float)(0.089019679316328 / -0.016958780164980), 5.05f},
    {-3.353001113951400e-04f, (float)(7.147062196813336e-04 / -3.353001113951400e-04), 5.35f},
    {-0.003702722457147f, (float)(0.005465945471933 / -0.003702722457147), 5.35f}};

A2C_HD float rsq(float x) { return eam::rsq_est(x); }

// Position of r in the tables: interval k and local coordinate u in [0, 1),
// computed once per quadrature point and shared by every function evaluated
// there.  Outside [1, 6) A ("far") k is clamped into the table so the reads
// stay in bounds and their results are replaced: from 6 A on by the
// exponential tails, below 1 A by NaN (no physical configuration comes that
// close -- the nearest Pd-H distance is 1.9 A -- and the non-finite
// objective makes the caller fall back to the FP64 path).
struct Pos {
  int k;
  float u;
  bool far;
};
__device__ __forceinline__ Pos tab_pos(float r) {
  const float xx = fmaf(r, INVH, -R0 * INVH);
  Pos p;
  p.k = min(max((int)xx, 0), NT - 1);
  p.u = __builtin_amdgcn_fractf(xx);
  p.far = !(fabsf(xx - 0.5f * NT) < 0.5f * NT);
  return p;
}
// value of a cubic row {c0, c1, c2, c3}
A2C_HD float cubic(const float4 c, float u) { return fmaf(u, fmaf(u, fmaf(u, c.w, c.z), c.y), c.x); }
// value and d/du of a cubic row (Horner with derivative: 5 FMAs)
A2C_HD void cubic_vd(const float4 c, float u, float& v, float& du) {
  const float v1 = fmaf(u, c.w, c.z);
  const float v2 = fmaf(u, v1, c.y);
  const float d2 = fmaf(u, c.w, v1);
  v = fmaf(u, v2, c.x);
  du = fmaf(u, d2, v2);
}
// value of a derivative row {c1, 2 c2, 3 c3, 0} (d/du of a cubic row)
A2C_HD float quad(const float4 c, float u) { return fmaf(u, fmaf(u, c.z, c.y), c.x); }
// exponential tail of function w (its slope is TAIL[w][1] times the value);
// NaN below the table (see tab_pos)
__device__ __forceinline__ float tail(int w, float r) {
  return r >= R1 ? TAIL[w][0] * __expf(TAIL[w][1] * (r - TAIL[w][2])) : __builtin_nanf("");
}

// value of table w at r (tails beyond the table; NaN below it)
__device__ __forceinline__ float tab_v(const float4* __restrict__ tab, int w, float r) {
  const Pos p = tab_pos(r);
  if (!p.far) return cubic(tab[w * NT + p.k], p.u);
  return tail(w, r);
}
// f_H(r) = 11.0025 exp(-1.30927 r) (potential.cpp:105-119; the exponential
// tail past 5.35 A continues the same function to 1e-13), evaluated without a
// table as 11.0025 * 2^(K r), K = -1.30927 log2(e) split into FP32 hi and lo
// parts, with the rounding of K r carried into a first-order correction: the
// value is within about an ulp of FP32 and costs one transcendental and five
// FMA-class instructions instead of a 16-byte LDS lookup.  NaN below 1 A, as
// the tables (see tab_pos).  Its slope is FH_K times the value.
constexpr double FH_K = -1.30927;
constexpr double LOG2E = 1.4426950408889634074;
constexpr float FH_C = 11.0025f;
constexpr float FH_KHI = (float)(FH_K * LOG2E);
constexpr float FH_KLO = (float)(FH_K * LOG2E - (double)FH_KHI);
constexpr float FH_KF = (float)FH_K;
constexpr float LN2F = 0.69314718055994530942f;
__device__ __forceinline__ float fH_exp(float r) {
  const float e = FH_KHI * r;
  const float el = fmaf(FH_KLO, r, fmaf(FH_KHI, r, -e));
  const float v = FH_C * __builtin_amdgcn_exp2f(e) * fmaf(el, LN2F, 1.0f);
  return r >= R0 ? v : __builtin_nanf("");
}
__device__ __forceinline__ Site load_site(const double* __restrict__ X, int s) {
  const double4 v = *reinterpret_cast<const double4*>(X + 4 * (size_t)s);
  return {{v.x, v.y, v.z}, v.w};
}
// d = q_i - image(q_j) in FP64, rounded to FP32 (geometry held in registers)
__device__ __forceinline__ void pair_vec32(const Image& g, const Site& a, const Site& b, float d[3]) {
  double dd[3];
  image_vec(g, a.q, b.q, dd);
#pragma unroll
  for (int c = 0; c < 3; ++c) d[c] = (float)dd[c];
}
// d = q_i - image(q_j) in FP64, rounded to FP32
__device__ __forceinline__ void pair_vec32(const LatDev& S, const Site& a, const Site& b, float d[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double qj = b.q[c];
    if (S.periodic[c]) qj = qj - S.box[c] * rint((qj - a.q[c]) * S.ibox[c]);
    d[c] = (float)(a.q[c] - qj);
  }
}

__device__ __forceinline__ void stage_tables(float4* lds, const float4* __restrict__ g, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) lds[i] = g[i];
  __syncthreads();
}
// Gradient passes need f_Pd only through f_Pd', staged as derivative rows
// {c1, 2 c2, 3 c3, 0}; the pair tables stay cubic; f_H is evaluated directly.
// LDS layout of the gradient passes: G_FPD (f_Pd'), G_PHPD, G_PHPDH, G_PHH,
// NT rows each (32 KB).
enum { G_FPD = 0, G_PHPD = 1, G_PHPDH = 2, G_PHH = 3, NGTAB = 4 };
__device__ __forceinline__ void stage_grad_tables(float4* lds, const float4* __restrict__ g) {
  for (int i = threadIdx.x; i < NGTAB * NT; i += blockDim.x) {
    const int w = i / NT, k = i - w * NT;
    const int src = w == G_FPD ? T_FPD : w + 1;  // T_PHPD, T_PHPDH, T_PHH follow T_FH in the global tables
    const float4 c = g[src * NT + k];
    lds[i] = w == G_FPD ? make_float4(c.y, 2.0f * c.z, 3.0f * c.w, 0.0f) : c;
  }
  __syncthreads();
}

// ---------------------------------------------------------------- density
// Sum of the table-w density over the 12 points of one pair.
__device__ __forceinline__ float pair_density(const float4* tab, int w, const float d[3], float ai, float aj) {
  const float D2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  const float bi = D2 + ai * ai, bj = D2 + aj * aj;
  float acc = 0.0f;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float ti = 2.0f * ai * d[c], tj = 2.0f * aj * d[c];
    const float r2[4] = {bi + ti, bi - ti, bj - tj, bj + tj};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float x = fmaxf(r2[q], 1e-12f);
      acc += tab_v(tab, w, x * rsq(x));
    }
  }
  return acc;
}

__global__ __launch_bounds__(TB) void k_density32(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l,
                                                  const float4* __restrict__ gtab) {
  __shared__ float4 tab[2 * NT];  // f_Pd, f_H
  stage_tables(tab, gtab, 2 * NT);
  const int blk = xcd_block();
  const LatDev& S = lats[b2l[blk]];
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
  const float ai = SQ6F * (float)a.s;
  double rho = 0.0;
  const int np = LP.cnt[row];
  for (int t = 0; t < np; ++t) {
    const int j = LP.idx[(size_t)t * LP.rows + row];
    const Site b = load_site(X, j);
    float d[3];
    pair_vec32(S, a, b, d);
    rho += (double)pair_density(tab, T_FPD, d, ai, SQ6F * (float)b.s);
  }
  const int nhn = LH.cnt[row];
  for (int t = 0; t < nhn; ++t) {
    const int h = LH.idx[(size_t)t * LH.rows + row];
    const Site b = load_site(X, S.npd + h);
    float d[3];
    pair_vec32(S, a, b, d);
    rho += xo[h] * (double)pair_density(tab, T_FH, d, ai, SQ6F * (float)b.s);
  }
  rho *= QW;
  S.rho[s] = rho;
  const double xs = pd ? 1.0 : xo[row];
  const eam::VD F = pd ? eam::F_Pd_vd(rho) : eam::F_H_vd(rho);
  S.aux[s] = make_float2((float)F.d, (float)xs);
  S.emb[s] = xs * F.v;
}

// ---------------------------------------------------------------- gradient
// Pair kinds: 0 Pd-Pd, 1 Pd-H (site Pd), 2 H-Pd (site H), 3 H-H.
// Per point: the pair energy phi(r) and cu = h dE/dr (h = 0.01 A, the table
// step; callers scale their per-pair sums by 1/h once) of the pair's share
// of the objective, dE/dr = F'_i f_j'(r) + F'_j f_i'(r) + phi'(r) (f_k: the
// density function of site k's species).  One table position serves all
// three functions.
template <int KIND>
__device__ __forceinline__ void point_coef(const float4* tab, float r, float Fi, float Fj, float& phi, float& cu) {
  constexpr int WP = KIND == 0 ? G_PHPD : (KIND == 3 ? G_PHH : G_PHPDH);    // LDS table of phi
  constexpr int TP = KIND == 0 ? T_PHPD : (KIND == 3 ? T_PHH : T_PHPDH);    // its tail
  const Pos p = tab_pos(r);
  float dphi;
  cubic_vd(tab[WP * NT + p.k], p.u, phi, dphi);
  // h f_H'(r) (h = 1/INVH, the table step): f_H' = FH_K f_H
  const float hdfh = KIND == 0 ? 0.0f : (FH_KF / INVH) * fH_exp(r);
  if (KIND == 0) {
    cu = fmaf(Fi + Fj, quad(tab[G_FPD * NT + p.k], p.u), dphi);
  } else if (KIND == 3) {
    cu = fmaf(Fi + Fj, hdfh, dphi);
  } else {
    const float Fpd = KIND == 1 ? Fi : Fj;  // F' of the Pd site multiplies f_H'
    const float Fh = KIND == 1 ? Fj : Fi;   // F' of the H site multiplies f_Pd'
    cu = fmaf(Fpd, hdfh, fmaf(Fh, quad(tab[G_FPD * NT + p.k], p.u), dphi));
  }
  if (p.far) {
    phi = tail(TP, r);
    const float dp = TAIL[TP][1] * phi;
    float c;
    if (KIND == 0) {
      c = fmaf(Fi + Fj, TAIL[T_FPD][1] * tail(T_FPD, r), dp);
    } else if (KIND == 3) {
      c = fmaf(Fi + Fj, hdfh * INVH, dp);
    } else {
      const float Fpd = KIND == 1 ? Fi : Fj;
      const float Fh = KIND == 1 ? Fj : Fi;
      c = fmaf(Fpd, hdfh * INVH, fmaf(Fh, TAIL[T_FPD][1] * tail(T_FPD, r), dp));
    }
    cu = c * (1.0f / INVH);
  }
}

struct PairSums {
  float pe;     // sum of phi over the 12 points
  float g[3];   // sum of (c/|r|) r
  float gs;     // sum over site-i points of (c/|r|) r . xi1 / sqrt(3)
};

template <int KIND>
__device__ __forceinline__ PairSums pair_grad(const float4* tab, const float d[3], float ai, float aj, float Fi,
                                              float Fj) {
  const float D2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  const float bi = D2 + ai * ai, bj = D2 + aj * aj;
  float su = 0.0f, ui = 0.0f, pe = 0.0f, ti[3], tj[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float t1 = 2.0f * ai * d[c], t2 = 2.0f * aj * d[c];
    // site-i points: r = d +- ai e_c ; site-j points: r = d -+ aj e_c
    const float r2[4] = {bi + t1, bi - t1, bj - t2, bj + t2};
    float u[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float x = fmaxf(r2[q], 1e-12f);
      const float rinv = rsq(x);
      float phi, cc;
      point_coef<KIND>(tab, x * rinv, Fi, Fj, phi, cc);
      pe += phi;
      u[q] = cc * rinv;
    }
    ti[c] = u[0] - u[1];
    tj[c] = u[2] - u[3];
    ui += u[0] + u[1];
    su += (u[0] + u[1]) + (u[2] + u[3]);
  }
  PairSums p;
  p.pe = pe;
#pragma unroll
  for (int c = 0; c < 3; ++c) p.g[c] = INVH * fmaf(d[c], su, ai * ti[c] - aj * tj[c]);
  p.gs = INVH * fmaf(d[0], ti[0], fmaf(d[1], ti[1], fmaf(d[2], ti[2], ai * ui)));
  return p;
}

__global__ __launch_bounds__(TB) void k_grad32(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l,
                                               const float4* __restrict__ gtab) {
  __shared__ float4 tab[NGTAB * NT];
  stage_grad_tables(tab, gtab);
  const int blk = xcd_block();
  const LatDev& S = lats[b2l[blk]];
  const int lb = blk - S.blk0;
  const int s = lb * TB + threadIdx.x;
  const int N = S.npd + S.nh;
  const double* __restrict__ X = S.X;
  const double* __restrict__ xo = S.x;
  const float2* __restrict__ aux = S.aux;
  double fs = 0.0;
  if (s < N) {
    const bool pd = s < S.npd;
    const int row = pd ? s : s - S.npd;
    const Ell LP = pd ? S.pdpd : S.hpd;
    const Ell LH = pd ? S.pdh : S.hh;
    const Site a = load_site(X, s);
    const float ai = SQ6F * (float)a.s;
    const float Fi = aux[s].x;
    const double xi = pd ? 1.0 : xo[row];
    double e = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0, gs = 0.0;
    const int np = LP.cnt[row];
    for (int t = 0; t < np; ++t) {
      const int j = LP.idx[(size_t)t * LP.rows + row];
      const Site b = load_site(X, j);
      const float2 nb = aux[j];
      float d[3];
      pair_vec32(S, a, b, d);
      const float aj = SQ6F * (float)b.s;
      const PairSums p = pd ? pair_grad<0>(tab, d, ai, aj, Fi, nb.x) : pair_grad<2>(tab, d, ai, aj, Fi, nb.x);
      e += p.pe; g0 += p.g[0]; g1 += p.g[1]; g2 += p.g[2]; gs += p.gs;
    }
    const int nhn = LH.cnt[row];
    for (int t = 0; t < nhn; ++t) {
      const int h = LH.idx[(size_t)t * LH.rows + row];
      const Site b = load_site(X, S.npd + h);
      const float2 nb = aux[S.npd + h];
      float d[3];
      pair_vec32(S, a, b, d);
      const float aj = SQ6F * (float)b.s;
      const PairSums p = pd ? pair_grad<1>(tab, d, ai, aj, Fi, nb.x) : pair_grad<3>(tab, d, ai, aj, Fi, nb.x);
      const double w = xo[h];  // occupancy of the H neighbor
      e += w * p.pe; g0 += w * p.g[0]; g1 += w * p.g[1]; g2 += w * p.g[2]; gs += w * p.gs;
    }
    const double T = S.T;
    const double V = S.emb[s] + 0.5 * QW * xi * e;
    const double sc = QW * xi / T;
    double* __restrict__ G = S.G;
    G[4 * (size_t)s + 0] = sc * g0;
    G[4 * (size_t)s + 1] = sc * g1;
    G[4 * (size_t)s + 2] = sc * g2;
    G[4 * (size_t)s + 3] = SQ6 * sc * gs - 3.0 * KB * xi / a.s;
    fs = V / T - 3.0 * KB * xi * log(a.s);
  }
  // block reduction in the (now free) table memory
  __syncthreads();
  double* red = reinterpret_cast<double*>(tab);
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
// Each unordered pair {s, j} is evaluated once, by its owner:
//   own(s, j) = (s < j) XOR ((s ^ j) & 1),
// which gives every site about half of each of its lists.  Every row is split
// at neighbor-build time into a compact owned half and a compact received half
// (same order as the row), so each lane loops over its own pairs only.  The
// owner adds its own share and writes the partner's share into the partner's
// received slot; a gather kernel adds the received shares in FP64.  Each
// buffer entry is written by exactly one lane, so results are deterministic.

// The owner passes read the EAM functions from cubic tables.  The Pd functions
// stand on a uniform grid in s = |r|^2: a node's s is D2 + a^2 +- 2 a d_c (linear
// in what differs between the nodes of a pair), so the table coordinate of a node
// is one addition, and dE/ds = (dE/dr) / (2 |r|) is the factor every gradient term
// needs -- no square root and no division per node.  h = 0.5025 / 14 puts their
// switch radii 5.0 and 5.05 A on grid nodes (25 and 25.5025 A^2); SNT intervals
// from S0 reach past 36 A^2.  phi_PdH and phi_HH have rows in r, 1/160 A apart from
// 156/160 A (their switch radius 5.35 A is a grid node): exponentials are steepest
// at short distances, where steps in s are the longest in r, and a node of an H
// pair has r at hand from f_H.
// Rows: values (S_FPD, the density pass) and slopes (S_DFPD) interpolate at
// the Chebyshev points; the pair functions (S_PHPD, R_PH*) integrate the quadratic
// interpolating their slope, so value and slope come from one row.  Below 1.8 A
// the quadratic in s is coarser for phi_Pd than the Hermite tables in r: Pd-Pd
// pairs with a node there are evaluated node by node from those.
// f_H = 11.0025 exp(-1.30927 |r|) is evaluated directly: |r| and the
// exponential cost fewer clocks (8 for each transcendental) than one more
// 16-byte row gathered from LDS (~12 clocks of the whole CU's LDS, which the
// two other rows of a Pd-H node already keep busy).
// Every function's error is held to that of the Hermite tables in r
// (tests/test_pass_tables.py).
// A node's coordinate is x = SINV s + SB, and f_H's s = SH x + S0; the rows are built on
// the grid that the first two floats define.  The four are floats near 14 / 0.5025
// and 683 - 25.5025 SINV that invert each other to 4e-10 (rounded apart: 1e-7 of
// every s, a bias of all values); the radii are 2e-5 of a row off their nodes.
constexpr float SINV = 27.860683f, SB = -27.517103f, SH = 0.035892874f, S0 = 0.9876679f;
constexpr double SH64 = 1.0 / (double)SINV, S064 = -(double)SB / (double)SINV;
static_assert((double)SH - SH64 < 1e-9 * SH64 && SH64 - (double)SH < 1e-9 * SH64 &&
                  (double)S0 + (double)SB * SH < 1e-9 && (double)S0 + (double)SB * SH > -1e-9,
              "SH and S0 invert SINV and SB");
constexpr float SLO = 1.0f, SHI = 36.0f;  // nodes the tables serve: [1, 6) A
constexpr float SLO_PHPD = 1.8f * 1.8f;   // and phi_Pd's rows in s
template <int KIND>
constexpr float s_lo() { return KIND == 0 ? SLO_PHPD : SLO; }
constexpr int SNT = 977;
constexpr float RINV = 160.0f, RB = -156.0f;
constexpr int RNT = 806;
constexpr int S_BASE = NTAB * NT;  // first row of these tables after those in r
enum { S_FPD = 0, S_DFPD = SNT, S_PHPD = 2 * SNT, R_PHPDH = 3 * SNT, R_PHH = R_PHPDH + RNT, S_ROWS = R_PHH + RNT };
enum { P_DFPD = 0, P_PHPD = SNT, P_PHPDH = 2 * SNT, P_PHH = P_PHPDH + RNT, P_ROWS = P_PHH + RNT };  // staged by the gradient pass
static_assert(S064 < 1.0 && S064 + (SNT - 1) * SH64 > 36.0, "the grid covers [1, 36] A^2");
static_assert((RNT - 1 - (double)RB) / (double)RINV > 6.0, "the grid covers [1, 6] A");

// Table coordinates and displacement squares of one pair.  12-point rule: the
// nodes of site i have s = bi +- 2 ai d_c, of site j bj -+ 2 aj d_c.
// inside(): every node lies in [1, 6) A; the largest |2 a d_c| bounds them.
struct Nodes12 {
  float xi, xj, gi, gj, lo, hi;  // ti = gi d_c, tj = gj d_c
  __device__ __forceinline__ Nodes12(const float d[3], float ai, float aj) {
    const float D2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    const float bi = fmaf(ai, ai, D2), bj = fmaf(aj, aj, D2);
    const float ei = 2.0f * ai, ej = 2.0f * aj;
    const float m = fmaxf(fmaxf(fabsf(d[0]), fabsf(d[1])), fabsf(d[2]));
    lo = fminf(fmaf(-fabsf(ei), m, bi), fmaf(-fabsf(ej), m, bj));
    hi = fmaxf(fmaf(fabsf(ei), m, bi), fmaf(fabsf(ej), m, bj));
    xi = fmaf(bi, SINV, SB);
    xj = fmaf(bj, SINV, SB);
    gi = ei * SINV;
    gj = ej * SINV;
  }
};
// Gauss-Hermite rule: s = D2 + 3 s^2 |a|^2 + 2 sqrt(3) s (a . d).
struct Nodes27 {
  float x0, n1, t[3], lo, hi;
  __device__ __forceinline__ Nodes27(const float d[3], float sd) {
    const float D2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    const float s3 = 3.0f * sd * sd, tt = 2.0f * GHZF * sd;
    lo = hi = D2;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float e = tt * fabsf(d[c]);
      lo += fminf(s3 - e, 0.0f);
      hi += s3 + e;
      t[c] = tt * SINV * d[c];
    }
    x0 = fmaf(D2, SINV, SB);
    n1 = s3 * SINV;
  }
};
template <int KIND>
__device__ __forceinline__ bool inside(float lo, float hi) { return lo >= s_lo<KIND>() && hi < SHI; }

// The nodes of a pair one at a time, for the pairs with a node outside.
// x(k): table coordinate of node k; w, off: its weight and displacement.
template <int RULE>
struct Edge {
  static constexpr int N = RULE == GH3 ? 27 : 12;
  float d[3], ai, aj, sd, off[3], w;
  int end;  // 12-point rule: the site that moves (0: i, 1: j)
  __device__ __forceinline__ Edge(const float* dd, float si, float sj)
      : d{dd[0], dd[1], dd[2]}, ai(SQ6F * si), aj(SQ6F * sj), sd(sqrtf(si * si + sj * sj)), w(1.0f), end(0) {}
  __device__ __forceinline__ float x(int k) {
    if (RULE == GH3) {
      const int a0 = k % 3 - 1, a1 = (k / 3) % 3 - 1, a2 = k / 9 - 1;
      w = ghwf(a0) * ghwf(a1) * ghwf(a2);
      off[0] = GHZF * sd * (float)a0;
      off[1] = GHZF * sd * (float)a1;
      off[2] = GHZF * sd * (float)a2;
    } else {
      end = k >= 6;
      const float a = (k & 1 ? -1.0f : 1.0f) * (end ? aj : ai);
      const int c = (k >> 1) % 3;
      off[0] = c == 0 ? a : 0.0f;
      off[1] = c == 1 ? a : 0.0f;
      off[2] = c == 2 ? a : 0.0f;
    }
    float s = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
#pragma unroll
    for (int c = 0; c < 3; ++c) s = fmaf(off[c], fmaf(2.0f, d[c], off[c]), s);
    return fmaf(s, SINV, SB);
  }
};

// f_H / 11.0025 at s, |r| and 1/|r|: 2^(K r), K = -1.30927 log2(e) split into
// FP32 hi and lo parts, with the rounding of K r carried into a first-order
// correction (within about an ulp of FP32).  Callers scale their sums.
A2C_HD float fH_s(float s, float& r, float& rinv) {
  rinv = rsq(s);
  r = s * rinv;
  const float e = FH_KHI * r;
  const float el = fmaf(FH_KLO, r, fmaf(FH_KHI, r, -e));
  return eam::exp2_est(e) * fmaf(el, LN2F, 1.0f);
}
// Row position of table coordinate x: interval k and u in [0, 1).
struct SPos {
  int k;
  float u;
};
A2C_HD SPos s_pos(float x) { return {(int)x, eam::fract(x)}; }
// s of a table coordinate, and whether the tables serve it (a pair with a
// node outside is evaluated node by node: the exponential tails from 6 A on,
// NaN below 1 A -- no physical configuration comes that close, and the
// non-finite objective makes the caller fall back to the FP64 path).
A2C_HD float s_of(float x) { return fmaf(x, SH, S0); }
__device__ __forceinline__ bool s_in(float s) { return s >= SLO && s < SHI; }
__device__ __forceinline__ float s_tail(int w, float s) {  // by s: at 36 the rounded radius may fall short of 6
  return s >= SHI ? TAIL[w][0] * __expf(TAIL[w][1] * (s * rsq(s) - TAIL[w][2])) : __builtin_nanf("");
}

// Densities at one node: f_Pd (tab: its value rows) and f_H / 11.0025, as wanted.
template <bool WANT_PD, bool WANT_H, bool IN>
__device__ __forceinline__ void node_dens(const float4* tab, float x, float& fpd, float& fh) {
  const float s = s_of(x);
  const bool in = IN || s_in(s);
  if (WANT_PD) {
    if (in) {
      const SPos p = s_pos(x);
      fpd = cubic(tab[p.k], p.u);
    } else {
      fpd = s_tail(T_FPD, s);
    }
  }
  if (WANT_H) {
    float r, ri;
    fh = in || s >= SHI ? fH_s(s, r, ri) : __builtin_nanf("");
  }
}

// Sums over a pair's nodes of two densities: the density of the neighbor's
// species (for this site) and of this site's species (for the neighbor); one
// sum when the species are the same.  NB_H / ME_H: neighbor / this site is an
// H site.  IN: every node is inside the tables.
template <bool NB_H, bool ME_H, bool IN>
__device__ __forceinline__ void pair_density2(const float4* tab, const Nodes12& q, const float d[3], float& sa, float& sb) {
  constexpr bool WP = !NB_H || !ME_H, WH = NB_H || ME_H;
  float sp = 0.0f, sh = 0.0f;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float ti = q.gi * d[c], tj = q.gj * d[c];
    const float x[4] = {q.xi + ti, q.xi - ti, q.xj - tj, q.xj + tj};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float fp = 0.0f, fh = 0.0f;
      node_dens<WP, WH, IN>(tab, x[k], fp, fh);
      if (WP) sp += fp;
      if (WH) sh += fh;
    }
  }
  sa = NB_H ? FH_C * sh : sp;
  sb = ME_H ? FH_C * sh : sp;
}
// The Gauss-Hermite sums: a rolled loop over the z offset a2, the 9 nodes of
// each plane unrolled (a fully unrolled 27 spills).
template <bool NB_H, bool ME_H, bool IN>
__device__ __forceinline__ void pair_density2_gh(const float4* tab, const Nodes27& q, float& sa, float& sb) {
  constexpr bool WP = !NB_H || !ME_H, WH = NB_H || ME_H;
  float sp = 0.0f, sh = 0.0f;
#pragma unroll 1
  for (int a2 = -1; a2 <= 1; ++a2) {
    const float base = q.x0 + q.n1 * (float)(a2 * a2) + (float)a2 * q.t[2];
    float pp = 0.0f, ph = 0.0f;
#pragma unroll
    for (int a1 = -1; a1 <= 1; ++a1) {
#pragma unroll
      for (int a0 = -1; a0 <= 1; ++a0) {
        const float w = ghwf(a0) * ghwf(a1);
        float fp = 0.0f, fh = 0.0f;
        node_dens<WP, WH, IN>(tab, base + q.n1 * (float)(a0 * a0 + a1 * a1) + (a0 * q.t[0] + a1 * q.t[1]), fp, fh);
        if (WP) pp += w * fp;
        if (WH) ph += w * fh;
      }
    }
    const float w2 = a2 ? 1.0f : 4.0f;
    if (WP) sp += w2 * pp;
    if (WH) sh += w2 * ph;
  }
  sa = NB_H ? FH_C * sh : sp;
  sb = ME_H ? FH_C * sh : sp;
}
template <int RULE, bool NB_H, bool ME_H>
__device__ __forceinline__ void pair_dens(const float4* tab, const float d[3], float as, float bs, float& mine,
                                          float& theirs) {
  bool in;
  if (RULE == GH3) {
    const Nodes27 q(d, sqrtf(as * as + bs * bs));
    in = inside<3>(q.lo, q.hi);
    if (in) pair_density2_gh<NB_H, ME_H, true>(tab, q, mine, theirs);
  } else {
    const Nodes12 q(d, SQ6F * as, SQ6F * bs);
    in = inside<3>(q.lo, q.hi);
    if (in) pair_density2<NB_H, ME_H, true>(tab, q, d, mine, theirs);
  }
  if (!in) {  // node by node, rolled (rare: a call would cost every pair the registers it keeps across it)
    constexpr bool WP = !NB_H || !ME_H, WH = NB_H || ME_H;
    Edge<RULE> q(d, as, bs);
    float sp = 0.0f, sh = 0.0f;
#pragma unroll 1
    for (int k = 0; k < Edge<RULE>::N; ++k) {
      float fp = 0.0f, fh = 0.0f;
      node_dens<WP, WH, false>(tab, q.x(k), fp, fh);
      sp += q.w * fp;
      sh += q.w * fh;
    }
    mine = NB_H ? FH_C * sh : sp;
    theirs = ME_H ? FH_C * sh : sp;
  }
}

struct Pair32 {
  float d[3], bs;
};

template <int RULE, bool BY_SITE, bool NB_H, bool ME_H>
__device__ __forceinline__ void dens_list(const float4* tab, const LatDev& S, const OwnerLane& ln, const Site& a,
                                          const Image& img, double wme, double& rho) {
  const Ell& L = ME_H ? (NB_H ? S.hh : S.hpd) : (NB_H ? S.pdh : S.pdpd);
  const Ell& P = ME_H ? (NB_H ? S.hh : S.pdh) : (NB_H ? S.hpd : S.pdpd);  // partner rows
  A2C_GLOBAL float* __restrict__ prb = gmem(reinterpret_cast<float*>(P.rbuf));
  const size_t prows = P.rows;
  const float as = (float)a.s;
  owned_pairs<NB_H, BY_SITE>(
      L, ln, S.kl32, S, [](int) { return 0.0f; },
      [&](const Site& b) {
        Pair32 p;
        pair_vec32(img, a, b, p.d);
        p.bs = (float)b.s;
        return p;
      },
      [&](const Pair32& p, float, double wj, int jl, int rv) {
        float mine, theirs;  // neighbor-species density (for me), my-species density (for the neighbor)
        pair_dens<RULE, NB_H, ME_H>(tab, p.d, as, p.bs, mine, theirs);
        rho += wj * (double)mine;
        // shares leave weighted by the sender's occupancy
        prb[(size_t)rv * prows + jl] = ME_H ? (float)(wme * (double)theirs) : theirs;
      });
}

// Bound by the vector ALUs and, as much, by the gathers' path through L1 (40^3
// cells: 70% and 88% of the time busy).  6 waves per SIMD: 80 VGPRs hold both
// rules' node blocks without spills.  40^3 cells, 12-point / Gauss-Hermite rule:
// 214 / 340 us with tables in |r|, sites in lattice order and the loads of a
// pair in its own turn, 146 / 260 us as it is (events of a2c_fe_time_eval).
template <int RULE, bool BY_SITE>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(6))) void k_dens_own(
    const LatDev* __restrict__ lats, const int32_t* __restrict__ ob2l, const float4* __restrict__ gtab) {
  __shared__ float4 tab[SNT];  // f_Pd (f_H is evaluated directly)
  const int w = xcd_block();
  const LatDev& S = lats[ob2l[w]];
  if (S.rule != RULE) return;  // whole workgroup: the other rule's instance serves this lattice
  stage16(tab, gtab + S_BASE + S_FPD, SNT);
  __syncthreads();
  const int K = S.kl32;
  const OwnerLane ln(S, w - S.owg0_32, K);
  if (ln.row >= ln.rows) return;  // whole lane groups
  const Image img = image_of(S);
  const int s = ln.pd ? ln.row : S.npd + ln.row;
  double wme;
  const Site a = own_site<BY_SITE>(S, ln, wme);
  double rho = 0.0;
  if (ln.pd) {
    dens_list<RULE, BY_SITE, false, false>(tab, S, ln, a, img, 1.0, rho);
    dens_list<RULE, BY_SITE, true, false>(tab, S, ln, a, img, 1.0, rho);
  } else {
    dens_list<RULE, BY_SITE, false, true>(tab, S, ln, a, img, wme, rho);
    dens_list<RULE, BY_SITE, true, true>(tab, S, ln, a, img, wme, rho);
  }
  rho = site_sum(rho, K);
  if (ln.ph == 0) gmem(S.rho)[s] = rho;
}

__global__ __launch_bounds__(TB) void k_dens_recv(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l,
                                                  int rq) {
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
    row_shares<RECV_RU_SCALAR, float>(L, row, ln.ph, ln.G, [&](float v) { rho += (double)v; });
  }
  rho = ln.sum(rho) + S.rho[s];
  if (ln.ph) return;
  rho *= S.rule == GH3 ? GHQW : QW;
  S.rho[s] = rho;
  const double xs = pd ? 1.0 : xo[row];
  const eam::VD F = pd ? eam::F_Pd_vd(rho) : eam::F_H_vd(rho);
  S.aux[s] = make_float2((float)F.d, (float)xs);
  S.emb[s] = xs * F.v;
}

struct PairSums2 {
  float pe;    // sum of phi
  float g[3];  // sum of (c/|r|) r           (q-gradient of site s; the partner gets -g)
  float gsi;   // site-s sigma term (x sqrt(6) QW x_s / T later)
  float gsj;   // partner sigma term
};

// One node: the pair energy phi and cu = SH dE/ds, E = F'_i f_j + F'_j f_i + phi
// (f_k: the density function of site k's species; KIND as in point_coef).
// FP multiplies f_Pd', FH f_H' / |r| (it carries FH_D).  tab: LDS rows of the
// gradient pass (P_*), gtab: the tables in r.
constexpr float FH_D = (float)(0.5 * SH64 * FH_K * 11.0025);
// phi_PdH or phi_HH (tab: its rows) at |r|^2 = s, r = sqrt(s) and ri = 1 / r rounded, and
// d/du.  The coordinate carries what r lost to rounding (0.5 ri (s - r^2)): the
// objective's noise, which ends the mixed phase of a relaxation, follows it.  40^3
// cells: +6 us, Gauss-Hermite +29; 64 lattices relaxed together 3,318 FP64 evaluations
// without it, 2,895 with it, 61.8 and 67.1 relaxations/s.
A2C_HD void phi_r(const float4* tab, float s, float r, float ri, float& v, float& d) {
  const float y = fmaf(r, RINV, fmaf((0.5f * RINV) * ri, fmaf(-r, r, s), RB));
  cubic_vd(tab[(int)y], eam::fract(y), v, d);
}
// phi_Pd from the Hermite rows in r (tab: all of its rows), and d/du
A2C_HD void phi_Pd_r(const float4* tab, float r, float& v, float& d) {
  const float y = fmaxf(fmaf(r, INVH, -R0 * INVH), 0.0f);
  cubic_vd(tab[(int)y], eam::fract(y), v, d);
}
template <int KIND, bool IN>
__device__ __forceinline__ void node_coef(const float4* tab, const float4* __restrict__ gtab, float x, float FP,
                                          float FH, float& phi, float& cu) {
  constexpr int TP = KIND == 0 ? T_PHPD : (KIND == 3 ? T_PHH : T_PHPDH);
  const float s = s_of(x);
  if (IN || s_in(s)) {
    const SPos p = s_pos(x);
    float d;
    if (KIND == 0) {
      if (IN || s >= SLO_PHPD) {
        cubic_vd(tab[P_PHPD + p.k], p.u, phi, cu);
      } else {
        const float ri = rsq(s);
        phi_Pd_r(gtab + T_PHPD * NT, s * ri, phi, d);
        cu = (0.5f * SH * INVH) * d * ri;
      }
    } else {
      float r, ri;
      const float fh = fH_s(s, r, ri);
      phi_r(tab + (KIND == 3 ? P_PHH : P_PHPDH), s, r, ri, phi, d);
      cu = fmaf(FH, fh, (0.5f * SH * RINV) * d) * ri;
    }
    if (KIND != 3) cu = fmaf(FP, cubic(tab[P_DFPD + p.k], p.u), cu);
  } else {
    const float ri = rsq(s);
    phi = s_tail(TP, s);
    float c = TAIL[TP][1] * phi;
    if (KIND != 3) c = fmaf(FP, TAIL[T_FPD][1] * s_tail(T_FPD, s), c);
    cu = 0.5f * SH * c * ri;
    if (KIND != 0) {
      float r1, r2;
      cu = fmaf(FH, s >= SHI ? fH_s(s, r1, r2) * ri : __builtin_nanf(""), cu);
    }
  }
}

// 12-point sums.  Site e's points are r = d +- a e_c with a = ai for the
// site and -aj for its partner.  With u = 2 SINV cu = (dE/dr) / |r| per node,
// T_c the difference of u between the two points of an axis, U_e their sum:
//   q-gradient  sum u r = d (U_i + U_j) + sum_e a T,
//   sigma terms d . T + a U (site i), its negative (partner).
// One axis of one site (2 nodes) per trip, the components rotating through
// d0 and h2: unrolled, the table rows of all nodes are in flight and their
// registers leave 4 waves per SIMD.
template <int KIND, bool IN>
__device__ __forceinline__ PairSums2 pair_grad2(const float4* tab, const float4* gtab, const Nodes12& n, const float d[3], float ai,
                                                float aj, float FP, float FH) {
  float pe = 0.0f, su = 0.0f, d0 = d[0], d1 = d[1], d2 = d[2], h0 = 0.0f, h1 = 0.0f, h2 = 0.0f;
  float a = ai, xb = n.xi, g = n.gi;
  PairSums2 p;
#pragma unroll 1
  for (int e = 0; e < 2; ++e) {
    float ue = 0.0f, se = 0.0f;
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
      const float t = g * d0;
      float phi0, phi1, u0, u1;
      node_coef<KIND, IN>(tab, gtab, xb + t, FP, FH, phi0, u0);
      node_coef<KIND, IN>(tab, gtab, xb - t, FP, FH, phi1, u1);
      pe += phi0 + phi1;
      const float T = u0 - u1;
      ue += u0 + u1;
      se = fmaf(d0, T, se);
      const float h = fmaf(a, T, h0), dt = d0;
      h0 = h1;
      h1 = h2;
      h2 = h;
      d0 = d1;
      d1 = d2;
      d2 = dt;
    }
    su += ue;
    p.gsj = -(2.0f * SINV) * fmaf(a, ue, se);
    if (e == 0) p.gsi = -p.gsj;
    a = -aj;
    xb = n.xj;
    g = -n.gj;
  }
  p.pe = pe;
  p.g[0] = (2.0f * SINV) * fmaf(d[0], su, h0);
  p.g[1] = (2.0f * SINV) * fmaf(d[1], su, h1);
  p.g[2] = (2.0f * SINV) * fmaf(d[2], su, h2);
  return p;
}

// Gauss-Hermite pair sums.  With u_k = w_k (c/|r_k|) and the node offsets
// a_k, n_k = |a_k|^2:  U = sum u, Va = sum u a, Wn = sum u n;
//   q-gradient  sum u r = d U + sqrt(3) s Va,
//   Sz = sum u (r . z) = sqrt(3) d . Va + 3 s Wn,  d/dsigma_k = Sz sigma_k / s.
template <int KIND, bool IN>
__device__ __forceinline__ PairSums2 pair_grad2_gh(const float4* tab, const float4* gtab, const Nodes27& q, const float d[3], float sd,
                                                   float si, float sj, float FP, float FH) {
  float pe = 0.0f, U = 0.0f, V0 = 0.0f, V1 = 0.0f, V2 = 0.0f, Wn = 0.0f;
#pragma unroll 1  // one z plane (9 nodes, unrolled) per trip, as in pair_density2_gh
  for (int a2 = -1; a2 <= 1; ++a2) {
    const float base = q.x0 + q.n1 * (float)(a2 * a2) + (float)a2 * q.t[2];
    float p9 = 0.0f, u9 = 0.0f, v0 = 0.0f, v1 = 0.0f, n9 = 0.0f;
#pragma unroll
    for (int a1 = -1; a1 <= 1; ++a1) {
#pragma unroll
      for (int a0 = -1; a0 <= 1; ++a0) {
        const int n = a0 * a0 + a1 * a1;
        const float w = ghwf(a0) * ghwf(a1);
        float phi, cc;
        node_coef<KIND, IN>(tab, gtab, base + q.n1 * (float)n + (a0 * q.t[0] + a1 * q.t[1]), FP, FH, phi, cc);
        p9 += w * phi;
        const float u = w * cc;
        u9 += u;
        if (a0) v0 += a0 * u;
        if (a1) v1 += a1 * u;
        if (n) n9 += n * u;
      }
    }
    const float w2 = a2 ? 1.0f : 4.0f;
    pe += w2 * p9;
    U += w2 * u9;
    V0 += w2 * v0;
    V1 += w2 * v1;
    V2 += (float)a2 * w2 * u9;
    Wn += w2 * fmaf((float)(a2 * a2), u9, n9);
  }
  PairSums2 p;
  p.pe = pe;
  const float sv = GHZF * sd;
  p.g[0] = (2.0f * SINV) * fmaf(d[0], U, sv * V0);
  p.g[1] = (2.0f * SINV) * fmaf(d[1], U, sv * V1);
  p.g[2] = (2.0f * SINV) * fmaf(d[2], U, sv * V2);
  const float sz = (2.0f * SINV) * fmaf(GHZF, fmaf(d[0], V0, fmaf(d[1], V1, d[2] * V2)), 3.0f * sd * Wn);
  p.gsi = sz * (si / sd);
  p.gsj = sz * (sj / sd);
  return p;
}

template <int RULE, int KIND>
__device__ __forceinline__ PairSums2 pair_grad(const float4* tab, const float4* gtab, const float d[3], float as, float bs, float Fi,
                                               float Fj) {
  const float FP = KIND == 0 ? Fi + Fj : (KIND == 1 ? Fj : Fi);           // F' of the H site multiplies f_Pd'
  const float FH = FH_D * (KIND == 3 ? Fi + Fj : (KIND == 1 ? Fi : Fj));  // F' of the Pd site f_H'
  PairSums2 p;
  bool in;
  if (RULE == GH3) {
    const float sd = sqrtf(as * as + bs * bs);
    const Nodes27 n(d, sd);
    in = inside<KIND>(n.lo, n.hi);
    if (in) p = pair_grad2_gh<KIND, true>(tab, gtab, n, d, sd, as, bs, FP, FH);
  } else {
    const float ai = SQ6F * as, aj = SQ6F * bs;
    const Nodes12 n(d, ai, aj);
    in = inside<KIND>(n.lo, n.hi);
    if (in) p = pair_grad2<KIND, true>(tab, gtab, n, d, ai, aj, FP, FH);
  }
  if (!in) {  // node by node, rolled, as in pair_dens
    Edge<RULE> q(d, as, bs);
    p = PairSums2{};
    float sz = 0.0f;
#pragma unroll 1
    for (int k = 0; k < Edge<RULE>::N; ++k) {
      float phi, u;
      node_coef<KIND, false>(tab, gtab, q.x(k), FP, FH, phi, u);
      p.pe = fmaf(q.w, phi, p.pe);
      u *= 2.0f * SINV * q.w;
      float ro = 0.0f;  // r . off
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float r = d[c] + q.off[c];
        p.g[c] = fmaf(u, r, p.g[c]);
        ro = fmaf(r, q.off[c], ro);
      }
      if (RULE == GH3) sz = fmaf(u, ro, sz);
      else if (q.end) p.gsj = fmaf(u, ro / q.aj, p.gsj);
      else p.gsi = fmaf(u, ro / q.ai, p.gsi);
    }
    if (RULE == GH3) {  // off = s z: d/dsigma_k = (sum u r . z) sigma_k / s
      p.gsi = sz * as / (q.sd * q.sd);
      p.gsj = sz * bs / (q.sd * q.sd);
    }
  }
  return p;
}

// Sums of one row's owned pairs.
struct Own {
  double e = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0, gs = 0.0;
};
template <int RULE, int KIND>
__device__ __forceinline__ void grad_list(const float4* tab, const float4* gtab, const LatDev& S, const OwnerLane& ln, const Site& a,
                                          float Fi, const Image& img, double wme, Own& o) {
  constexpr bool ME_H = KIND >= 2, NB_H = KIND & 1;
  const Ell& L = ME_H ? (NB_H ? S.hh : S.hpd) : (NB_H ? S.pdh : S.pdpd);
  const Ell& P = ME_H ? (NB_H ? S.hh : S.pdh) : (NB_H ? S.hpd : S.pdpd);  // partner rows
  A2C_GLOBAL float4* __restrict__ prb = gmem(reinterpret_cast<float4*>(P.rbuf));
  const size_t prows = P.rows;
  const float as = (float)a.s;
  const A2C_GLOBAL float2* aux = gmem((const float2*)S.aux) + (NB_H ? S.npd : 0);
  owned_pairs<NB_H>(
      L, ln, S.kl32, S, [=](int j) { return aux[j].x; },
      [&](const Site& b) {
        Pair32 p;
        pair_vec32(img, a, b, p.d);
        p.bs = (float)b.s;
        return p;
      },
      [&](const Pair32& q, float Fj, double wj, int jl, int rv) {
        const PairSums2 p = pair_grad<RULE, KIND>(tab, gtab, q.d, as, q.bs, Fi, Fj);
        o.e += wj * p.pe;
        o.g0 += wj * p.g[0];
        o.g1 += wj * p.g[1];
        o.g2 += wj * p.g[2];
        o.gs += wj * p.gsi;
        // the partner's share leaves weighted by the sender's occupancy
        float4 v = make_float4(-p.g[0], -p.g[1], -p.g[2], p.gsj);
        if (ME_H)
          v = make_float4((float)(wme * (double)v.x), (float)(wme * (double)v.y), (float)(wme * (double)v.z),
                          (float)(wme * (double)v.w));
        prb[(size_t)rv * prows + jl] = v;
      });
}

// Bound by what a pair moves: 8 B of list, ~50 B gathered through L1 and 16 B of
// share written (0.33 GB at 40^3 cells) keep the kernel at 246 us with its
// nodes taken out; with them 275 us (12-point rule; 364 us before the tables,
// the row order and the pipelined loads) and 535 us (Gauss-Hermite; 651 us), events of
// a2c_fe_time_eval.
template <int RULE, int TBO>
__global__ __launch_bounds__(TBO) __attribute__((amdgpu_waves_per_eu(TBO / 128))) void k_grad_own(
    const LatDev* __restrict__ lats, const int32_t* __restrict__ ob2l, int nblk, const float4* __restrict__ gtab) {
  __shared__ float4 tab[P_ROWS];
  stage16(tab, gtab + S_BASE + S_DFPD, P_ROWS);
  __syncthreads();
  const int w = xcd_block() * (TBO / TB) + __builtin_amdgcn_readfirstlane(threadIdx.x / TB);
  if (w >= nblk) return;
  const LatDev& S = lats[ob2l[w]];
  if (S.rule != RULE) return;  // the other rule's instance serves this lattice
  const int K = S.kl32;
  const OwnerLane ln(S, w - S.owg0_32, K);
  if (ln.row >= ln.rows) return;  // whole lane groups
  const Image img = image_of(S);
  const int s = ln.pd ? ln.row : S.npd + ln.row;
  const Site a = load_row(gmem((const double2*)S.qxy), gmem((const double2*)S.qzs), s);
  const float Fi = gmem((const float2*)S.aux)[s].x;
  Own o;
  if (ln.pd) {
    grad_list<RULE, 0>(tab, gtab, S, ln, a, Fi, img, 1.0, o);
    grad_list<RULE, 1>(tab, gtab, S, ln, a, Fi, img, 1.0, o);
  } else {
    const double wme = gmem((const double*)S.xrow)[ln.row];
    grad_list<RULE, 2>(tab, gtab, S, ln, a, Fi, img, wme, o);
    grad_list<RULE, 3>(tab, gtab, S, ln, a, Fi, img, wme, o);
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

__global__ __launch_bounds__(TB) void k_grad_recv(const LatDev* __restrict__ lats, const int32_t* __restrict__ b2l,
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
      row_shares<RECV_RU_WIDE, float4>(L, row, ln.ph, ln.G, [&](const float4& v) {
        g0 += v.x; g1 += v.y; g2 += v.z;
        gs += v.w;
      });
    }
    g0 = ln.sum(g0); g1 = ln.sum(g1); g2 = ln.sum(g2); gs = ln.sum(gs);
    const double xi = pd ? 1.0 : xo[row];
    const double sg = S.qzs[s].y;
    const double T = S.T;
    const bool gh = S.rule == GH3;
    const double qw = gh ? GHQW : QW, sq = gh ? 1.0 : SQ6;
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

}  // namespace

namespace {
// ---------------------------------------------------------------- tables
template <class Fn>
void fill_table(float4* out, Fn g) {
  const long double h = H64, eps = 1e-13L;
  for (int i = 0; i < NT; ++i) {
    const long double ra = (long double)R0 + i * h + eps, rb = (long double)R0 + (i + 1) * h - eps;
    const eam::VDT<long double> A = g(ra), B = g(rb);
    const long double c0 = A.v, c1 = h * A.d;
    const long double c2 = 3 * (B.v - A.v) - h * (2 * A.d + B.d);
    const long double c3 = 2 * (A.v - B.v) + h * (A.d + B.d);
    out[i] = make_float4((float)c0, (float)c1, (float)c2, (float)c3);
  }
}

// Rows of the tables in s: g gives a function's value and slope in |r|.  In
// the local coordinate u of an interval, the slope d/du is dg/dr h / (2 |r|).
struct Row {
  long double c[4] = {0, 0, 0, 0};
};
// polynomial through (u[i], y[i]), i < n, as monomials
Row through(const long double* u, const long double* y, int n) {
  long double c[4];
  for (int i = 0; i < n; ++i) c[i] = y[i];
  for (int j = 1; j < n; ++j)
    for (int i = n - 1; i >= j; --i) c[i] = (c[i] - c[i - 1]) / (u[i] - u[i - j]);
  Row m;
  for (int i = n - 1; i >= 0; --i) {
    for (int q = 3; q > 0; --q) m.c[q] = m.c[q - 1] - u[i] * m.c[q];
    m.c[0] = c[i] - u[i] * m.c[0];
  }
  return m;
}
enum { FIT_VALUE, FIT_SLOPE, FIT_BOTH };
// rows of the tables in s, or in r; g gives a function's value and slope in |r|
template <class Fn>
void fill_rows(float4* out, int rows, bool in_r, int fit, Fn g) {
  using LD = long double;
  const LD PI = 3.14159265358979323846264338327950288L;
  auto node = [&](int i, int n) { return 0.5L - 0.5L * cosl((2 * i + 1) * PI / (2.0L * n)); };
  for (int k = 0; k < rows; ++k) {
    auto at = [&](LD u) {
      const LD x = k + u, r = in_r ? (x - (LD)RB) / (LD)RINV : sqrtl((x - (LD)SB) / (LD)SINV);
      const eam::VDT<LD> v = g(r);
      return eam::VDT<LD>{v.v, v.d / (in_r ? (LD)RINV : 2 * r * (LD)SINV)};  // d/du
    };
    const int n = fit == FIT_BOTH ? 3 : 4;
    LD u[4], y[4];
    for (int i = 0; i < n; ++i) {
      u[i] = node(i, n);
      y[i] = fit == FIT_VALUE ? at(u[i]).v : at(u[i]).d;
    }
    Row m = through(u, y, n);
    if (fit == FIT_BOTH) {  // the slope's integral, with the value's mean over four points
      m = Row{{0, m.c[0], m.c[1] / 2, m.c[2] / 3}};
      for (int i = 0; i < 4; ++i) {
        const LD w = node(i, 4);
        y[i] = at(w).v - w * (m.c[1] + w * (m.c[2] + w * m.c[3]));
      }
      m.c[0] = (y[0] + y[1] + y[2] + y[3]) / 4;
    }
    out[k] = make_float4((float)m.c[0], (float)m.c[1], (float)m.c[2], (float)m.c[3]);
  }
}

}  // namespace

void host_tables_s(std::vector<float4>& t) {
  static const std::vector<float4> built = [] {  // once per process
    using LD = long double;
    std::vector<float4> u((size_t)S_ROWS);
    fill_rows(&u[S_FPD], SNT, false, FIT_VALUE, [](LD r) { return eam::f_Pd_vd<LD>(r); });
    fill_rows(&u[S_DFPD], SNT, false, FIT_SLOPE, [](LD r) { return eam::f_Pd_vd<LD>(r); });
    fill_rows(&u[S_PHPD], SNT, false, FIT_BOTH, [](LD r) { return eam::phi_Pd_vd<LD>(r, eam::f_Pd_vd<LD>(r)); });
    fill_rows(&u[R_PHPDH], RNT, true, FIT_BOTH, [](LD r) { return eam::phi_morse_vd<0, LD>(r); });
    fill_rows(&u[R_PHH], RNT, true, FIT_BOTH, [](LD r) { return eam::phi_morse_vd<1, LD>(r); });
    return u;
  }();
  t.insert(t.end(), built.begin(), built.end());
}

void host_tables(std::vector<float4>& t) {
  static const std::vector<float4> built = [] {  // once per process (~0.4 ms of long-double work)
    using LD = long double;
    std::vector<float4> u((size_t)NTAB * NT, make_float4(0.f, 0.f, 0.f, 0.f));
    fill_table(&u[T_FPD * NT], [](LD r) { return eam::f_Pd_vd<LD>(r); });
    fill_table(&u[T_FH * NT], [](LD r) { return eam::f_H_vd<LD>(r); });
    fill_table(&u[T_PHPD * NT], [](LD r) { return eam::phi_Pd_vd<LD>(r, eam::f_Pd_vd<LD>(r)); });
    fill_table(&u[T_PHPDH * NT], [](LD r) { return eam::phi_morse_vd<0, LD>(r); });
    fill_table(&u[T_PHH * NT], [](LD r) { return eam::phi_morse_vd<1, LD>(r); });
    return u;
  }();
  t = built;
}

// One EAM function (order of a2c_eam_tables) near r in [1, 6) A as the pair-once
// passes take it from the tables t (those in r, then these), value and slope in r,
// at the radius returned: what the FP32 table coordinate of r stands for.
double pass_eval32(const std::vector<float4>& t, int fn, double r0, double& v, double& d) {
  const float x = fmaf((float)(r0 * r0), SINV, SB);
  const double r_at = std::sqrt(((double)x - (double)SB) / (double)SINV);
  const SPos p = s_pos(x);
  const float4* u = &t[S_BASE];
  const float s = s_of(x);
  const double ds = 2.0 * SINV * r_at;  // of d/du in s
  float vf = 0.0f, df = 0.0f, r, ri;
  const float fh = fH_s(s, r, ri);
  if (fn == T_FH) {
    v = (double)FH_C * fh;
    d = FH_K * FH_C * fh;
    return r_at;
  }
  if (fn == T_FPD) {
    vf = cubic(u[S_FPD + p.k], p.u);
    df = cubic(u[S_DFPD + p.k], p.u);
    d = ds * df;
  } else if (fn == T_PHPD && s < SLO_PHPD) {
    phi_Pd_r(&t[T_PHPD * NT], r, vf, df);
    d = (double)INVH * df;
  } else if (fn == T_PHPD) {
    cubic_vd(u[S_PHPD + p.k], p.u, vf, df);
    d = ds * df;
  } else {
    phi_r(u + (fn == T_PHPDH ? R_PHPDH : R_PHH), s, r, ri, vf, df);
    d = (double)RINV * df;
  }
  v = vf;
  return r_at;
}

int build_tables(a2c_fe_ctx* c) {
  DeviceTables t;
  A2C_HIP(c, device_tables(c->desc.device, &t));
  c->dtab = t.t32;
  if (!c->daux) A2C_HIP(c, dmalloc(&c->daux, sizeof(float2) * std::max(c->N, 1)));
  return A2C_OK;
}

namespace {
// The tables of k_grad_own allow two workgroups per CU whatever their size: 512
// lanes give every SIMD 4 waves (40^3 cells: 264 us against 416 us with 256
// lanes and 2 waves).  With fewer units than two per CU the smaller
// workgroups spread over more CUs (14^3 cells, Gauss-Hermite rule: 53 against
// 56 us; 12-point rule 34 against 33 us).
constexpr int GRAD_WIDE_UNITS = 512;
template <int RULE>
void launch_grad_own(const Launch& L) {
  if (L.onblk >= GRAD_WIDE_UNITS)
    hipLaunchKernelGGL((k_grad_own<RULE, 512>), dim3((L.onblk + 1) / 2), dim3(512), 0, L.stream, L.lats, L.ob2l,
                       L.onblk, L.tab);
  else
    hipLaunchKernelGGL((k_grad_own<RULE, 256>), dim3(L.onblk), dim3(256), 0, L.stream, L.lats, L.ob2l, L.onblk,
                       L.tab);
}
}  // namespace

int run_eval32(const Launch& L, Timing* tm) {
  if (L.mixed_full && L.rules == (1 << A2C_QUAD_R12)) {  // every pair from both ends (12-point rule only)
    if (tm) tm->mark(L.stream, "density32");
    if (L.nblk > 0) {
      hipLaunchKernelGGL(k_density32, dim3(L.nblk), dim3(TB), 0, L.stream, L.lats, L.b2l, L.tab);
      if (hipGetLastError() != hipSuccess) return A2C_EHIP;
    }
    if (tm) tm->mark(L.stream, "grad32");
    if (L.nblk > 0) {
      hipLaunchKernelGGL(k_grad32, dim3(L.nblk), dim3(TB), 0, L.stream, L.lats, L.b2l, L.tab);
      if (hipGetLastError() != hipSuccess) return A2C_EHIP;
    }
  } else if (L.nblk > 0) {
    const bool fold = fold_rows(L);
    if (!fold) {
      if (tm) tm->mark(L.stream, "rows");
      if (run_rows(L)) return A2C_EHIP;
    }
    if (tm) tm->mark(L.stream, "dens_own");
    auto own = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(L.onblk), dim3(TB), 0, L.stream, L.lats, L.ob2l, L.tab);
    };
    if (L.onblk > 0 && (L.rules & (1 << A2C_QUAD_R12)))
      fold ? own(k_dens_own<A2C_QUAD_R12, true>) : own(k_dens_own<A2C_QUAD_R12, false>);
    if (L.onblk > 0 && (L.rules & (1 << GH3))) fold ? own(k_dens_own<GH3, true>) : own(k_dens_own<GH3, false>);
    if (hipGetLastError() != hipSuccess) return A2C_EHIP;
    if (tm) tm->mark(L.stream, "dens_recv");
    hipLaunchKernelGGL(k_dens_recv, dim3(L.nblk * L.rq), dim3(TB), 0, L.stream, L.lats, L.b2l, L.rq);
    if (hipGetLastError() != hipSuccess) return A2C_EHIP;
    if (tm) tm->mark(L.stream, "grad_own");
    if (L.onblk > 0 && (L.rules & (1 << A2C_QUAD_R12))) launch_grad_own<A2C_QUAD_R12>(L);
    if (L.onblk > 0 && (L.rules & (1 << GH3))) launch_grad_own<GH3>(L);
    if (hipGetLastError() != hipSuccess) return A2C_EHIP;
    if (tm) tm->mark(L.stream, "grad_recv");
    hipLaunchKernelGGL(k_grad_recv, dim3(L.nblk * L.rq), dim3(TB), 0, L.stream, L.lats, L.b2l, L.rq);
    if (hipGetLastError() != hipSuccess) return A2C_EHIP;
    if (tm) tm->mark(L.stream, nullptr);
    return A2C_OK;
  }
  if (tm) tm->mark(L.stream, "final_sum");
  if (int rc = run_final_sum(L)) return rc;
  if (tm) tm->mark(L.stream, nullptr);
  return A2C_OK;
}

}  // namespace a2c

// Host-only: the FP32 tables of the mixed path (no GPU needed).  Layout: 5
// tables (f_Pd, f_H, phi_Pd, phi_PdH, phi_H) x 500 intervals x {c0,c1,c2,c3},
// interval k covers r in [1 + 0.01 k, 1 + 0.01 (k+1)), value
// c0 + u(c1 + u(c2 + u c3)) with u = (r - 1)/0.01 - k.
extern "C" int a2c_eam_tables(float* out, int32_t cap) {
  std::vector<float4> t;
  a2c::host_tables(t);
  const int n = (int)t.size() * 4;
  if (out && cap >= n) std::memcpy(out, t.data(), sizeof(float) * n);
  return n;
}
