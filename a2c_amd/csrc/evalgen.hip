// Objective, gradient, density and chemical potential of a context with a
// general model: a tabulated potential (a2c_fe_set_potential_*) and/or a
// node table (a2c_fe_set_quadrature).  The reference's loop nests
// (minimizer.cpp:140-157 and :162-351 for the objective and gradient,
// :588-802 for the chemical potential, electrondensity.cpp:12-56 for the
// density) with the EAM functions and the rule as data.  Density and gradient
// take each pair once, at its owner, like the passes of the built-in rules
// (row order and shares: Ell and LatDev):
//
//   k_gen_rows       row-order copies of the state and the occupancy
//   k_gen_dens_own   owned pairs' density: own sums, shares to the partners
//   k_gen_dens_recv  rho, F(rho), F'(rho), the embedding energy
//   k_gen_grad_own   owned pairs' energy and coefficient c = F'_i f_j' +
//                    F'_j f_i' + phi' at each node, both ends' q- and
//                    sigma-gradient
//   k_gen_grad_recv  gradient, the site's share of f, block sums and f
//   k_gen_chem       per H site over its full lists: dV/dx_a + the correction
//                    terms, gamma, cap
//
// A node k of a 6-D table puts the pair vector at r_k = d + a_i xi1_k -
// a_j xi2_k with a = sqrt(2) sigma, so dr_k/dsigma_i = sqrt(2) xi1_k; a
// relative-coordinate rule (Gauss-Hermite) at r_k = d + s z_k with
// s^2 = sigma_i^2 + sigma_j^2, dr_k/dsigma_i = (sigma_i / s) z_k.  Both ends of
// a pair see the same average when the table is swap-symmetric (enforced
// when it is set), which the reference's pair terms assume.
//
// Precision: FP64 throughout, or (MIXED) the pair terms of each node in
// FP32 from FP32 pieces of the r-functions, summed per pair in FP32 and per
// site in FP64.  F(rho) and F'(rho) are FP64 in both.
#include <cmath>
#include <type_traits>

#include "eam64.hpp"
#include "fe_internal.hpp"
#include "pair_rows.hpp"

namespace a2c {
namespace {

constexpr int TB = SITE_BLOCK;
constexpr double SQ2 = 1.4142135623730950488;

__device__ __forceinline__ Site load_site(const double* __restrict__ X, int s) {
  const double4 v = *reinterpret_cast<const double4*>(X + 4 * (size_t)s);
  return {{v.x, v.y, v.z}, v.w};
}
__device__ __forceinline__ void pair_vec(const Image& g, const Site& a, const Site& b, double d[3]) {
  image_vec(g, a.q, b.q, d);
}

// ------------------------------------------------------------ functions
// Embedding functions in FP64: closed forms or pieces (the cubic in the local
// coordinate u of piece k; past the last node the end tangent).
__device__ __forceinline__ eam::VD emb_vd(const GenFn& F, const double4* __restrict__ tab, double x) {
  const double p = x * F.ih;
  int k = (int)p;
  if (k < 0) k = 0;
  if (k >= F.n - 1) return {F.yend + F.dend * (x - (double)(F.n - 1) / F.ih), F.dend};
  const double u = p - (double)k;
  const double4 c = tab[F.off + k];
  return {c.x + u * (c.y + u * (c.z + u * c.w)), (c.y + u * (2.0 * c.z + u * 3.0 * c.w)) * F.ih};
}
template <int POT>
__device__ __forceinline__ double F_val(const GenDev& g, bool pd, double rho) {
  if (POT == 0) return pd ? eam::F_Pd(rho) : eam::F_H(rho);
  return emb_vd(g.fn[pd ? GEN_F_PD : GEN_F_H], g.tab, rho).v;
}
template <int POT, int DM>
__device__ __forceinline__ double F_der(const GenDev& g, bool pd, double rho, double eps) {
  if (DM == A2C_DERIV_FD) return (F_val<POT>(g, pd, rho + eps) - F_val<POT>(g, pd, rho - eps)) / (2.0 * eps);
  if (POT == 0) return pd ? eam::F_Pd_vd(rho).d : eam::F_H_vd(rho).d;
  return emb_vd(g.fn[pd ? GEN_F_PD : GEN_F_H], g.tab, rho).d;
}

// |r| and 1/|r| from |r|^2, to the last place or so: the hardware estimate of
// 1/sqrt and Newton steps; at 0, infinity and NaN the limits (r = x, and the
// estimate itself).
__device__ __forceinline__ void root(double x, double& r, double& ri) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  ri = fma(y * e, fma(e, 0.375, 0.5), y);
  r = x * ri;
  r = fma(0.5 * ri, fma(-r, r, x), r);
  if (!(x > 0.0 && x < __builtin_huge_val())) r = x, ri = y;
}
__device__ __forceinline__ void root(float x, float& r, float& ri) {
  const float y = __builtin_amdgcn_rsqf(x);
  r = x * y;
  r = fmaf(0.5f * y, fmaf(-r, r, x), r);
  ri = fmaf(y, fmaf(-r, y, 1.0f), y);
  if (!(x > 0.0f && x < __builtin_huge_valf())) r = x, ri = y;
}

// A radius located in the r-functions' table: the row of its interval, the
// coordinate u in it, and whether it lies inside (past the table's end the
// functions are 0).
template <class R>
struct At;
template <>
struct At<double> {
  const A2C_GLOBAL double2* row;
  double r, ri, u, ih;
  bool in;
  // the Hermite piece of two nodes: c0, c1 from the first, c3 = s0 + s1 - 2 (y1
  // - y0), c2 = (y1 - y0) - s0 - c3
  template <int SLOT>
  __device__ __forceinline__ eam::VD vd() const {
    const double2 a = row[SLOT], b = row[GEN_NS + SLOT];
    const double dy = b.x - a.x, c3 = fma(-2.0, dy, a.y + b.y), c2 = (dy - a.y) - c3;
    return {fma(u, fma(u, fma(u, c3, c2), a.y), a.x), fma(u, fma(u, 3.0 * c3, c2 + c2), a.y) * ih};
  }
};
template <>
struct At<float> {
  const A2C_GLOBAL float4* row;
  float r, ri, u, ih;
  bool in;
  template <int SLOT>
  __device__ __forceinline__ eam::VDT<float> vd() const {
    const float4 c = row[SLOT];
    return {fmaf(u, fmaf(u, fmaf(u, c.w, c.z), c.y), c.x), fmaf(u, fmaf(u, 3.0f * c.w, c.z + c.z), c.y) * ih};
  }
};

// r-functions by slot: density f and pair phi (stored as r phi).  POT 0 in
// FP64: the closed forms; otherwise the table.
template <int POT, class R>
struct RFun {
  using E = std::conditional_t<sizeof(R) == 8, double2, float4>;
  static constexpr bool CLOSED = POT == 0 && sizeof(R) == 8;
  const A2C_GLOBAL E* row;
  int last;  // the last interval
  R ih;
  __device__ __forceinline__ explicit RFun(const GenDev& g) {
    if constexpr (sizeof(R) == 8) row = gmem((const E*)g.r64.row), last = g.r64.n - 2, ih = g.r64.ih;
    else row = gmem((const E*)g.r32.row), last = g.r32.n - 2, ih = (R)g.r32.ih;
  }
  __device__ __forceinline__ At<R> at(R r, R ri) const {
    At<R> a;
    a.r = r;
    a.ri = ri;
    if (CLOSED) return a;
    const R p = r * ih;
    const int k = max((int)p, 0);
    a.u = p - (R)k;
    a.ih = ih;
    a.in = k <= last;
    a.row = row + (size_t)GEN_NS * min(k, last);  // no branch around the loads: several nodes' are in flight together
    return a;
  }
  template <int SLOT>
  __device__ __forceinline__ eam::VDT<R> vd(const At<R>& a) const {
    if constexpr (CLOSED) {
      if constexpr (SLOT == GEN_S_RHO_PD) return eam::f_Pd_vd(a.r);
      else if constexpr (SLOT == GEN_S_RHO_H) return eam::f_H_vd(a.r);
      else if constexpr (SLOT == GEN_S_RPHI_PD) return eam::phi_Pd_vd(a.r, eam::f_Pd_vd(a.r));
      else return eam::phi_morse_vd<SLOT == GEN_S_RPHI_PDH ? 0 : 1>(a.r);
    } else {
      eam::VDT<R> z = a.template vd<SLOT>();
      if (!a.in) z = {R(0), R(0)};
      if constexpr (SLOT == GEN_S_RHO_PD || SLOT == GEN_S_RHO_H) return z;
      const R phi = z.v * a.ri;
      return {phi, (z.d - phi) * a.ri};  // (r phi)' = phi + r phi'
    }
  }
  template <int SLOT>
  __device__ __forceinline__ R val(const At<R>& a) const {
    if constexpr (CLOSED) {
      if constexpr (SLOT == GEN_S_RHO_PD) return eam::f_Pd(a.r);
      else if constexpr (SLOT == GEN_S_RHO_H) return eam::f_H(a.r);
      else if constexpr (SLOT == GEN_S_RPHI_PD) return eam::phi_Pd(a.r);
      else return eam::phi_morse<SLOT == GEN_S_RPHI_PDH ? 0 : 1>(a.r);
    } else {
      return vd<SLOT>(a).v;
    }
  }
};

// One node of a pair as the derivative mode wants it: the radius, and for the
// reference's central differences the radii eps to either side.
template <int POT, int DM, class R>
struct NodeR {
  RFun<POT, R> fun;
  At<R> c, hi, lo;
  R h;  // 1 / (2 eps)
  __device__ __forceinline__ NodeR(const RFun<POT, R>& f, R r, R ri, R eps) : fun(f), c(f.at(r, ri)) {
    if (DM == A2C_DERIV_FD) {
      hi = f.at(r + eps, R(1) / (r + eps));
      lo = f.at(r - eps, R(1) / (r - eps));
      h = R(2) * eps;
    }
  }
  template <int SLOT>
  __device__ __forceinline__ eam::VDT<R> vd() const {
    if (DM == A2C_DERIV_FD)
      return {fun.template val<SLOT>(c), (fun.template val<SLOT>(hi) - fun.template val<SLOT>(lo)) / h};
    return fun.template vd<SLOT>(c);
  }
};

// The rule's nodes staged in LDS as R, 8 to a node: xi1 (or z), xi2, w, 0.
extern __shared__ __align__(16) unsigned char gen_lds[];
template <class R>
__device__ __forceinline__ const R* stage_nodes(const GenDev& g) {
  R* nd = reinterpret_cast<R*>(gen_lds);
  for (int i = threadIdx.x; i < g.K * 8; i += blockDim.x) nd[i] = (R)g.nodes[i];
  __syncthreads();
  return nd;
}
template <class R>
size_t node_bytes(const GenDev& g) {
  return sizeof(R) * 8 * (size_t)g.K;
}

// Nodes of a pair: r_k = d + a xi1_k - b xi2_k; dr_k/dsigma of the first site
// is fi xi1_k, of the second -fj xi2_k (6-D nodes) or fj z_k (relative ones).
template <class R>
struct PairFrame {
  R d[3], a, b;
  R fi, fj;
};
template <class R>
__device__ __forceinline__ PairFrame<R> frame(const GenDev& g, const double d[3], double si, double sj) {
  PairFrame<R> f;
  f.d[0] = (R)d[0];
  f.d[1] = (R)d[1];
  f.d[2] = (R)d[2];
  if (g.rel) {
    const double s = sqrt(si * si + sj * sj);
    f.a = (R)s;
    f.b = R(0);
    f.fi = (R)(si / s);
    f.fj = (R)(sj / s);
  } else {
    f.a = (R)(SQ2 * si);
    f.b = (R)(SQ2 * sj);
    f.fi = f.fj = (R)SQ2;
  }
  return f;
}
template <class R>
__device__ __forceinline__ R node_r2(const PairFrame<R>& f, const R* n, R r[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) r[c] = f.d[c] + f.a * n[c] - f.b * n[3 + c];
  return r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
}

struct GenPair {
  double d[3], s;
};
__device__ __forceinline__ GenPair gen_pair(const Image& img, const Site& a, const Site& b) {
  GenPair p;
  pair_vec(img, a, b, p.d);
  p.s = b.s;
  return p;
}

__global__ __launch_bounds__(TB) void k_gen_rows(const LatDev* __restrict__ lat) {
  const LatDev& S = *lat;
  const int s = xcd_block() * TB + threadIdx.x;
  copy_row(S, s);
}

// ------------------------------------------------------------ density
template <int POT, class R, bool BY_SITE, bool NB_H, bool ME_H>
__device__ __forceinline__ void dens_list(const LatDev& S, const GenDev& g, const RFun<POT, R>& fun, const R* nd,
                                          const OwnerLane& ln, int KL, const Site& a, const Image& img, double wme,
                                          double& rho) {
  constexpr int NB = NB_H ? GEN_S_RHO_H : GEN_S_RHO_PD, ME = ME_H ? GEN_S_RHO_H : GEN_S_RHO_PD;
  const Ell& L = ME_H ? (NB_H ? S.hh : S.hpd) : (NB_H ? S.pdh : S.pdpd);
  const Ell& P = ME_H ? (NB_H ? S.hh : S.pdh) : (NB_H ? S.hpd : S.pdpd);  // partner rows
  A2C_GLOBAL double* __restrict__ share = gmem(reinterpret_cast<double*>(P.rbuf));
  const size_t prows = P.rows;
  owned_pairs<NB_H, BY_SITE>(
      L, ln, KL, S, [](int) { return 0.0f; }, [&](const Site& b) { return gen_pair(img, a, b); },
      [&](const GenPair& p, float, double wj, int jl, int rv) {
        const PairFrame<R> f = frame<R>(g, p.d, a.s, p.s);
        R mine = R(0), theirs = R(0);
#pragma unroll 2  // two nodes' gathers in flight
        for (int k = 0; k < g.K; ++k) {
          const R* n = nd + 8 * k;
          R r[3], rn, ri;
          root(node_r2(f, n, r), rn, ri);
          const At<R> at = fun.at(rn, ri);
          mine += n[6] * fun.template val<NB>(at);
          if (NB != ME) theirs += n[6] * fun.template val<ME>(at);
        }
        if (NB == ME) theirs = mine;
        rho += wj * (double)mine;
        share[(size_t)rv * prows + jl] = wme * (double)theirs;
      });
}

// 16^3 cells, tabulated potential, 12 nodes, FP64: full lists, one lane per site
// 306 us, this 77 us; the gradient pass 727 and 118 us.  Bound by the L1: a node's
// gathers (two 16-byte words per function) touch a line per lane.  5^3 cells (memory
// latency): 62 us with a branch around the table's end, 52 without, 41 with two
// nodes in flight; more nodes only take registers.
template <int POT, class R, bool BY_SITE>
__global__ __launch_bounds__(TB) void k_gen_dens_own(const LatDev* __restrict__ lat, GenDev g, int KL) {
  const R* nd = stage_nodes<R>(g);
  const LatDev& S = *lat;
  const OwnerLane ln(S, __builtin_amdgcn_readfirstlane(xcd_block()), KL);
  if (ln.row >= ln.rows) return;  // whole lane groups
  const RFun<POT, R> fun(g);
  const Image img = image_of(S);
  const int s = ln.pd ? ln.row : S.npd + ln.row;
  double wme;
  const Site a = own_site<BY_SITE>(S, ln, wme);
  double rho = 0.0;
  if (ln.pd) {
    dens_list<POT, R, BY_SITE, false, false>(S, g, fun, nd, ln, KL, a, img, 1.0, rho);
    dens_list<POT, R, BY_SITE, true, false>(S, g, fun, nd, ln, KL, a, img, 1.0, rho);
  } else {
    dens_list<POT, R, BY_SITE, false, true>(S, g, fun, nd, ln, KL, a, img, wme, rho);
    dens_list<POT, R, BY_SITE, true, true>(S, g, fun, nd, ln, KL, a, img, wme, rho);
  }
  rho = site_sum(rho, KL);
  if (ln.ph == 0) gmem(S.epair)[s] = rho;
}

// by_site: rho, F' and the embedding energy in site order (the chemical
// potential and a caller's density), else in row order (the gradient pass).
template <int POT, int DM>
__global__ __launch_bounds__(TB) void k_gen_dens_recv(const LatDev* __restrict__ lat, GenDev g, double eps,
                                                      int by_site) {
  const LatDev& S = *lat;
  const int v = xcd_block(), rq = S.rl;
  const RecvLane ln(S, v / rq, v % rq);
  const int s = ln.s;
  if (s >= S.npd + S.nh) return;
  const bool pd = s < S.npd;
  const int row = pd ? s : s - S.npd;
  double rho = 0.0;
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const Ell& L = pd ? (side ? S.pdh : S.pdpd) : (side ? S.hh : S.hpd);
    row_shares<RECV_RU_SCALAR, double>(L, row, ln.ph, ln.G, [&](double v) { rho += v; });
  }
  rho = ln.sum(rho) + S.epair[s];
  if (ln.ph) return;
  const double F = F_val<POT>(g, pd, rho);
  const int o = !by_site ? s : pd ? site_of_row(row, S.npd) : S.npd + site_of_row(row, S.nh);
  S.rho[o] = rho;
  S.Fp[o] = F_der<POT, DM>(g, pd, rho, eps);
  S.emb[o] = pd ? F : S.xrow[row] * F;
}

// ------------------------------------------------------------ gradient
// Kinds: 0 Pd-Pd, 1 Pd site / H neighbor, 2 H site / Pd neighbor, 3 H-H.
// phi and c = dE/dr of one node; FP multiplies f_Pd', FH f_H'.
template <int POT, int DM, class R, int KIND>
__device__ __forceinline__ void node_terms(const NodeR<POT, DM, R>& n, R FP, R FH, R& phi, R& c) {
  constexpr int PHI = KIND == 0 ? GEN_S_RPHI_PD : KIND == 3 ? GEN_S_RPHI_H : GEN_S_RPHI_PDH;
  const eam::VDT<R> p = n.template vd<PHI>();
  phi = p.v;
  c = p.d;
  if (KIND != 3) c += FP * n.template vd<GEN_S_RHO_PD>().d;
  if (KIND != 0) c += FH * n.template vd<GEN_S_RHO_H>().d;
}

struct Own {
  double e = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0, gs = 0.0;
};
template <int POT, int DM, class R, int KIND>
__device__ __forceinline__ void grad_list(const LatDev& S, const GenDev& g, const RFun<POT, R>& fun, const R* nd,
                                          const OwnerLane& ln, int KL, const Site& a, double Fi, const Image& img,
                                          double wme, R eps, Own& o) {
  constexpr bool ME_H = KIND >= 2, NB_H = KIND & 1;
  const Ell& L = ME_H ? (NB_H ? S.hh : S.hpd) : (NB_H ? S.pdh : S.pdpd);
  const Ell& P = ME_H ? (NB_H ? S.hh : S.pdh) : (NB_H ? S.hpd : S.pdpd);  // partner rows
  A2C_GLOBAL double4* __restrict__ share = gmem(reinterpret_cast<double4*>(P.rbuf));
  const size_t prows = P.rows;
  const A2C_GLOBAL double* Fp = gmem((const double*)S.Fp) + (NB_H ? S.npd : 0);
  owned_pairs<NB_H>(
      L, ln, KL, S, [=](int j) { return Fp[j]; }, [&](const Site& b) { return gen_pair(img, a, b); },
      [&](const GenPair& q, double Fj, double wj, int jl, int rv) {
        const PairFrame<R> f = frame<R>(g, q.d, a.s, q.s);
        // a site's density takes the partner's f
        const R FP = KIND == 0 ? (R)Fi + (R)Fj : KIND == 1 ? (R)Fj : (R)Fi;
        const R FH = KIND == 3 ? (R)Fi + (R)Fj : KIND == 1 ? (R)Fi : (R)Fj;
        R pe = R(0), px = R(0), py = R(0), pz = R(0), ps = R(0), pt = R(0);
#pragma unroll 1
        for (int k = 0; k < g.K; ++k) {
          const R* n = nd + 8 * k;
          R r[3], rn, ri, phi, c;
          root(node_r2(f, n, r), rn, ri);
          node_terms<POT, DM, R, KIND>(NodeR<POT, DM, R>(fun, rn, ri, eps), FP, FH, phi, c);
          const R w = n[6];
          pe += w * phi;
          const R u = w * c * ri;
          px += u * r[0];
          py += u * r[1];
          pz += u * r[2];
          ps += u * (r[0] * n[0] + r[1] * n[1] + r[2] * n[2]);
          pt -= u * (r[0] * n[3] + r[1] * n[4] + r[2] * n[5]);
        }
        if (g.rel) pt = ps;
        o.e += wj * (double)pe;
        o.g0 += wj * (double)px;
        o.g1 += wj * (double)py;
        o.g2 += wj * (double)pz;
        o.gs += wj * (double)(ps * f.fi);
        // the partner's share leaves weighted by the sender's occupancy
        share[(size_t)rv * prows + jl] =
            make_double4(-wme * (double)px, -wme * (double)py, -wme * (double)pz, wme * (double)(pt * f.fj));
      });
}

template <int POT, int DM, class R>
__global__ __launch_bounds__(TB) void k_gen_grad_own(const LatDev* __restrict__ lat, GenDev g, double eps, int KL) {
  const R* nd = stage_nodes<R>(g);
  const LatDev& S = *lat;
  const OwnerLane ln(S, __builtin_amdgcn_readfirstlane(xcd_block()), KL);
  if (ln.row >= ln.rows) return;  // whole lane groups
  const RFun<POT, R> fun(g);
  const Image img = image_of(S);
  const int s = ln.pd ? ln.row : S.npd + ln.row;
  const Site a = load_row(gmem((const double2*)S.qxy), gmem((const double2*)S.qzs), s);
  const double Fi = gmem((const double*)S.Fp)[s];
  Own o;
  if (ln.pd) {
    grad_list<POT, DM, R, 0>(S, g, fun, nd, ln, KL, a, Fi, img, 1.0, (R)eps, o);
    grad_list<POT, DM, R, 1>(S, g, fun, nd, ln, KL, a, Fi, img, 1.0, (R)eps, o);
  } else {
    const double wme = gmem((const double*)S.xrow)[ln.row];
    grad_list<POT, DM, R, 2>(S, g, fun, nd, ln, KL, a, Fi, img, wme, (R)eps, o);
    grad_list<POT, DM, R, 3>(S, g, fun, nd, ln, KL, a, Fi, img, wme, (R)eps, o);
  }
  o.e = site_sum(o.e, KL);
  o.g0 = site_sum(o.g0, KL);
  o.g1 = site_sum(o.g1, KL);
  o.g2 = site_sum(o.g2, KL);
  o.gs = site_sum(o.gs, KL);
  if (ln.ph != 0) return;
  gmem(S.gown)[s] = make_double4(o.g0, o.g1, o.g2, o.gs);
  gmem(S.epair)[s] = o.e;
}

__global__ __launch_bounds__(TB) void k_gen_grad_recv(const LatDev* __restrict__ lat) {
  const LatDev& S = *lat;
  const int v = xcd_block(), rq = S.rl;
  const RecvLane ln(S, v / rq, v % rq);
  const int s = ln.s;
  double fs = 0.0, sl = 0.0;
  if (s < S.npd + S.nh) {
    const bool pd = s < S.npd;
    const int row = pd ? s : s - S.npd;
    const size_t site = pd ? site_of_row(row, S.npd) : S.npd + site_of_row(row, S.nh);
    double4 gr = ln.ph ? make_double4(0.0, 0.0, 0.0, 0.0) : S.gown[s];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const Ell& L = pd ? (side ? S.pdh : S.pdpd) : (side ? S.hh : S.hpd);
      row_shares<RECV_RU_WIDE, double4>(L, row, ln.ph, ln.G, [&](const double4& v) {
        gr.x += v.x; gr.y += v.y; gr.z += v.z;
        gr.w += v.w;
      });
    }
    gr = make_double4(ln.sum(gr.x), ln.sum(gr.y), ln.sum(gr.z), ln.sum(gr.w));
    if (ln.ph == 0) {
      const double xi = pd ? 1.0 : S.xrow[row];
      const double sg = S.qzs[s].y;
      const double T = S.T, sc = xi / T;
      const double V = S.emb[s] + xi * S.epair[s];  // owned pairs carry their full energy (minimizer.cpp:169-286)
      double* __restrict__ G = S.G + 4 * site;  // the caller's: 8-byte aligned
      gr = make_double4(sc * gr.x, sc * gr.y, sc * gr.z, sc * gr.w - 3.0 * KB * xi / sg);
      G[0] = gr.x;
      G[1] = gr.y;
      G[2] = gr.z;
      G[3] = gr.w;
      fs = V / T - 3.0 * KB * xi * log(sg);
      sl = site_slope(S, site, gr.x, gr.y, gr.z, gr.w);
    }
  }
  finish_objective(S, ln, fs, sl);
}

// ------------------------------------------------------------ chemical potential
// minimizer.cpp:588-802 per H site a (FP64): F_H(rho_a) + the H-Pd and H-H
// pair sums with the neighbor's F' + the correction terms (corr from
// k_chem_pre), gamma = ln(x/(1-x)) + sum/(kB T) + 1.5 for 0 < x < 1, capped.
template <int POT>
__global__ __launch_bounds__(TB) void k_gen_chem(const LatDev* __restrict__ lat, GenDev g,
                                                 const double* __restrict__ corr, double ch0, double ch1, double ch2,
                                                 double ch3, double gamma_bd, double* __restrict__ gamma,
                                                 int32_t* __restrict__ full) {
  const double* nd = stage_nodes<double>(g);
  const LatDev& S = *lat;
  const int a = blockIdx.x * TB + threadIdx.x;
  if (a >= S.nh || full[a] == 1) return;  // fully occupied reservoir: gamma untouched
  const RFun<POT, double> fun(g);
  const Image img = image_of(S);
  const double* __restrict__ X = S.X;
  const double* __restrict__ xo = S.x;
  const double* __restrict__ Fp = S.Fp;
  const int s = S.npd + a;
  const Site si = load_site(X, s);
  const double T = S.T;
  const int K = g.K;
  double sum = F_val<POT>(g, false, S.rho[s]);
  const double n = (double)S.hpd.cnt[a];
  double Xa = 0.0;
  const int nhh = S.hh.cnt[a];
  for (int t = 0; t < nhh; ++t) Xa += xo[S.hh.idx[(size_t)t * S.hh.rows + a]];
  sum += 0.5 * T * ch0 * (ch1 * n * n + 2.0 * ch2 * n * Xa + ch3 * Xa * Xa);
  for (int side = 0; side < 2; ++side) {  // H-Pd (:679-698), then H-H (:701-719)
    const Ell L = side == 0 ? S.hpd : S.hh;
    const int m = L.cnt[a];
    for (int t = 0; t < m; ++t) {
      const int jl = L.idx[(size_t)t * L.rows + a];
      const int j = side == 0 ? jl : S.npd + jl;
      const Site b = load_site(X, j);
      double d[3];
      pair_vec(img, si, b, d);
      const PairFrame<double> f = frame<double>(g, d, si.s, b.s);
      double sf = 0.0, sp = 0.0;
      for (int k = 0; k < K; ++k) {
        const double* n = nd + 8 * k;
        double r[3], rn, ri;
        root(node_r2(f, n, r), rn, ri);
        const At<double> at = fun.at(rn, ri);
        sf += n[6] * fun.template val<GEN_S_RHO_H>(at);
        sp += n[6] * (side == 0 ? fun.template val<GEN_S_RPHI_PDH>(at) : fun.template val<GEN_S_RPHI_H>(at));
      }
      const double term = Fp[j] * sf + sp + corr[j];
      sum += side == 0 ? term : xo[jl] * term;
    }
  }
  const double x = xo[a];
  const double raw = (x > 0.0 && x < 1.0) ? log(x / (1.0 - x)) + sum / (KB * T) : 0.0;
  double gm = raw + 1.5;
  if (gm > gamma_bd) {
    gm = gamma_bd;
    if (x > 0.9999) full[a] = 1;
  }
  gamma[a] = gm;
}

// The kernel instance for (potential, derivative mode, precision).  The
// FP32 instances read the r-functions from FP32 pieces whatever the
// potential (the closed forms have pieces of their own, general.cpp) and F
// like the FP64 ones.  Central differences of step ~1e-5 are meaningless in
// FP32, so FD mode runs the FP64 instances in either precision.
template <template <int, int, class> class Pick>
auto pick(const GenDev& g, int deriv_mode, bool fp32) {
  const bool fd = deriv_mode == A2C_DERIV_FD, tab = g.pot == 1;
  if (fd) return tab ? Pick<1, A2C_DERIV_FD, double>::fn : Pick<0, A2C_DERIV_FD, double>::fn;
  if (fp32) return tab ? Pick<1, A2C_DERIV_ANALYTIC, float>::fn : Pick<0, A2C_DERIV_ANALYTIC, float>::fn;
  return tab ? Pick<1, A2C_DERIV_ANALYTIC, double>::fn : Pick<0, A2C_DERIV_ANALYTIC, double>::fn;
}
template <int P, int D, class R> struct DensK { static constexpr auto fn = k_gen_dens_own<P, R, false>; };
template <int P, int D, class R> struct DensFoldK { static constexpr auto fn = k_gen_dens_own<P, R, true>; };
template <int P, int D, class R> struct RecvK { static constexpr auto fn = k_gen_dens_recv<P, D>; };
template <int P, int D, class R> struct GradK { static constexpr auto fn = k_gen_grad_own<P, D, R>; };

bool general_fp32(int deriv_mode, bool fp32) { return fp32 && deriv_mode != A2C_DERIV_FD; }
size_t lds_bytes(const GenDev& g, int deriv_mode, bool fp32) {
  return general_fp32(deriv_mode, fp32) ? node_bytes<float>(g) : node_bytes<double>(g);
}

// Lanes per site: the mixed passes' table in either precision.  These kernels
// wait for gathers where the FP64 passes compute (16^3 cells, FP64, K = 1/2/4/8:
// 580/333/238/251 us).
int gen_lanes(int n) { return lanes_per_site(n, false); }

// rho, F(rho), F'(rho) and the embedding energy at the state of *dlat.
int run_density_gen(const LatDev* dlat, int npd, int nh, const GenDev& g, int deriv_mode, double eps, bool fp32,
                    bool by_site, hipStream_t st, Timing* tm) {
  if (npd + nh <= 0) return A2C_OK;
  const int nblk = site_blocks(npd + nh), KL = gen_lanes(npd + nh);
  const bool fold = nblk <= FOLD_BLOCKS;
  if (!fold) {
    if (tm) tm->mark(st, "rows");
    hipLaunchKernelGGL(k_gen_rows, dim3(nblk), dim3(TB), 0, st, dlat);
  }
  if (tm) tm->mark(st, "gen_dens_own");
  hipLaunchKernelGGL(fold ? pick<DensFoldK>(g, deriv_mode, fp32) : pick<DensK>(g, deriv_mode, fp32),
                     dim3(owner_units(npd, nh, KL)), dim3(TB), lds_bytes(g, deriv_mode, fp32), st, dlat, g, KL);
  if (tm) tm->mark(st, "gen_dens_recv");
  hipLaunchKernelGGL(pick<RecvK>(g, deriv_mode, fp32), dim3(nblk * recv_lanes(npd + nh)), dim3(TB), 0, st, dlat, g, eps, (int)by_site);
  return hipGetLastError() == hipSuccess ? A2C_OK : A2C_EHIP;
}

}  // namespace

int run_eval_gen(const LatDev* dlat, int npd, int nh, const GenDev& g, int deriv_mode, double eps, bool fp32,
                 hipStream_t st, Timing* tm) {
  if (npd + nh > 0) {
    const int nblk = site_blocks(npd + nh), KL = gen_lanes(npd + nh);
    if (int rc = run_density_gen(dlat, npd, nh, g, deriv_mode, eps, fp32, false, st, tm)) return rc;
    if (tm) tm->mark(st, "gen_grad_own");
    hipLaunchKernelGGL(pick<GradK>(g, deriv_mode, fp32), dim3(owner_units(npd, nh, KL)), dim3(TB),
                       lds_bytes(g, deriv_mode, fp32), st, dlat, g, eps, KL);
    if (tm) tm->mark(st, "gen_grad_recv");
    hipLaunchKernelGGL(k_gen_grad_recv, dim3(nblk * recv_lanes(npd + nh)), dim3(TB), 0, st, dlat);
    if (hipGetLastError() != hipSuccess) return A2C_EHIP;
    if (tm) tm->mark(st, nullptr);
    return A2C_OK;
  }
  if (tm) tm->mark(st, "final_sum");
  Launch L{};
  L.lats = dlat;
  L.nlat = 1;
  L.stream = st;
  if (int rc = run_final_sum(L)) return rc;
  if (tm) tm->mark(st, nullptr);
  return A2C_OK;
}

int launch_density_gen(a2c_fe_ctx* c, const double* dX) {
  if (int rc = sync_lattice(c, dX, c->dG, c->dF)) return rc;
  // the density feeding F' is FP64 in both precisions
  if (run_density_gen(c->dlat, c->desc.n_pd, c->desc.n_h, c->gen, c->desc.deriv_mode, c->desc.fd_eps, false, true,
                      c->stream, nullptr))
    return set_err(c, A2C_EHIP, "general density launch failed");
  return A2C_OK;
}

int launch_eval_gen(a2c_fe_ctx* c, const double* dX, double* dG, double* dF, bool timed, Timing* tm) {
  if (int rc = sync_lattice(c, dX, dG, dF)) return rc;
  if (run_eval_gen(c->dlat, c->desc.n_pd, c->desc.n_h, c->gen, c->desc.deriv_mode, c->desc.fd_eps,
                   c->desc.precision == A2C_PREC_MIXED, c->stream, timed ? tm : nullptr))
    return set_err(c, A2C_EHIP, "general eval launch failed");
  return A2C_OK;
}

int launch_chem_gen(a2c_fe_ctx* c, const double* dX, const double* coe_h, double gamma_bd, double* dgam,
                    int32_t* dfull, const double* dcorr) {
  (void)dX;  // the descriptor already points at dX (launch_density_gen)
  const int nh = c->desc.n_h;
  if (nh <= 0) return A2C_OK;
  hipLaunchKernelGGL(c->gen.pot == 1 ? k_gen_chem<1> : k_gen_chem<0>, dim3((nh + TB - 1) / TB), dim3(TB),
                     node_bytes<double>(c->gen), c->stream, (const LatDev*)c->dlat, c->gen, dcorr, coe_h[0], coe_h[1], coe_h[2], coe_h[3],
                     gamma_bd, dgam, dfull);
  A2C_HIP(c, hipGetLastError());
  return A2C_OK;
}

}  // namespace a2c
