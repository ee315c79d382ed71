// What the pair-owner passes of both precisions share: a site's state in row
// order, and the walk over a row's owned pairs.
#pragma once
#include "fe_internal.hpp"

namespace a2c {
namespace {

// n 16-byte words from global memory to LDS by the whole workgroup
__device__ __forceinline__ void stage16(void* lds, const void* g, int n) {
  uint4* __restrict__ d = reinterpret_cast<uint4*>(lds);
  const uint4* __restrict__ s = reinterpret_cast<const uint4*>(g);
  for (int i = threadIdx.x; i < n; i += blockDim.x) d[i] = s[i];
}

struct Site {
  double q[3];
  double s;
};
__device__ __forceinline__ Site load_row(const A2C_GLOBAL double2* __restrict__ qxy,
                                         const A2C_GLOBAL double2* __restrict__ qzs, int p) {
  const double2 a = qxy[p], b = qzs[p];
  return {{a.x, a.y, b.x}, b.y};
}

// the state and occupancy of site s to their place in row order; site 0's lane
// also clears the count of finished blocks
__device__ __forceinline__ void copy_row(const LatDev& S, int s) {
  if (s == 0) *S.done = 0;
  if (s >= S.npd + S.nh) return;
  const double4 v = reinterpret_cast<const double4*>(S.X)[s];
  const bool pd = s < S.npd;
  const int row = pd ? row_of_site(s, S.npd) : row_of_site(s - S.npd, S.nh);
  const int p = pd ? row : S.npd + row;
  S.qxy[p] = make_double2(v.x, v.y);
  S.qzs[p] = make_double2(v.z, v.w);
  if (!pd) S.xrow[row] = S.x[s - S.npd];
}

// A species' sites by row: the row-order copies, or (BY_SITE) the caller's
// site-order arrays.
template <bool BY_SITE, bool H>
struct RowState {
  const A2C_GLOBAL double2* __restrict__ qxy;
  const A2C_GLOBAL double2* __restrict__ qzs;
  const A2C_GLOBAL double* __restrict__ w;
  __device__ __forceinline__ explicit RowState(const LatDev& S)
      : qxy(gmem((const double2*)S.qxy) + (H ? S.npd : 0)),
        qzs(gmem((const double2*)S.qzs) + (H ? S.npd : 0)),
        w(gmem((const double*)S.xrow)) {}
  __device__ __forceinline__ Site site(int row) const { return load_row(qxy, qzs, row); }
  __device__ __forceinline__ double occ(int row) const { return w[row]; }
};
template <bool H>
struct RowState<true, H> {
  const A2C_GLOBAL double4* __restrict__ X;
  const A2C_GLOBAL double* __restrict__ x;
  int rows;
  __device__ __forceinline__ explicit RowState(const LatDev& S)
      : X(gmem(reinterpret_cast<const double4*>(S.X)) + (H ? S.npd : 0)), x(gmem(S.x)), rows(H ? S.nh : S.npd) {}
  __device__ __forceinline__ Site site(int row) const {
    const double4 v = X[site_of_row(row, rows)];
    return {{v.x, v.y, v.z}, v.w};
  }
  __device__ __forceinline__ double occ(int row) const { return x[site_of_row(row, rows)]; }
};

// A density pass that reads the site-order arrays writes the row-order copies
// for the passes behind it (and does the rest of k_rows' work): a launch less.
// It gathers from four times the lines, so only launches of up to FOLD_BLOCKS
// blocks of 256 sites do.  k_rows and density pass apart / together, mixed: 1,728
// sites 18.3 / 12.1 us, 21,952 sites 26.0 / 20.3, 46,656 sites 31.1 / 26.2, 110,592
// sites 47.8 / 45.3, 262,144 sites 90 / 111 (with ~2 us of timing events per
// launch).
constexpr int FOLD_BLOCKS = 256;
template <bool BY_SITE>
__device__ __forceinline__ Site own_site(const LatDev& S, const OwnerLane& ln, double& occ) {
  const int s = ln.pd ? ln.row : S.npd + ln.row;
  Site a;
  if (ln.pd) {
    a = RowState<BY_SITE, false>(S).site(ln.row);
    occ = 1.0;
  } else {
    const RowState<BY_SITE, true> h(S);
    a = h.site(ln.row);
    occ = h.occ(ln.row);
  }
  if (BY_SITE && ln.ph == 0) {
    gmem(S.qxy)[s] = make_double2(a.q[0], a.q[1]);
    gmem(S.qzs)[s] = make_double2(a.q[2], a.s);
    if (!ln.pd) gmem(S.xrow)[ln.row] = occ;
    if (s == 0) *S.done = 0;  // without Pd sites H row 0 has s = 0
  }
  return a;
}

// Owned pairs of one list of one row, K lanes per row.  Software pipeline: at
// a pair's turn the state of the next one and the index and slot of the one
// after it are requested, then the pair is evaluated and its share stored.
// Loads and stores complete in order on one counter, so a load requested
// after a store cannot be waited for without waiting for the store to reach
// memory; requested one pair earlier, every load is older than the stores
// still in flight (k_grad_own, 40^3 cells: 290 -> 261 us).  F(j): F' of
// neighbor row j; geom(b): the pair's geometry; eval(geometry, F'_j, w_j,
// neighbor row, received slot): the rest, w_j the occupancy of an H neighbor.
template <bool NB_H, bool BY_SITE = false, class LoadF, class Geom, class Eval>
__device__ __forceinline__ void owned_pairs(const Ell& L, const OwnerLane& ln, int K, const LatDev& S, LoadF F,
                                            Geom geom, Eval eval) {
  const size_t rows = L.rows, first = (size_t)ln.ph * rows + ln.row, step = (size_t)K * rows;
  const A2C_GLOBAL int32_t* __restrict__ oj = gmem((const int32_t*)L.oj) + first;
  const A2C_GLOBAL int32_t* __restrict__ orv = gmem((const int32_t*)L.orv) + first;
  const RowState<BY_SITE, NB_H> st(S);
  const int n = gmem((const int32_t*)L.ocnt)[ln.row];
  int t = ln.ph;
  if (t >= n) return;
  size_t e = t + K < n ? step : 0;  // past the row's end its last entry is requested again: no branch around
                                    // a load, or the waits behind it cover everything outstanding
  int j1 = oj[0], r1 = orv[0], j2 = oj[e], r2 = orv[e];
  Site b = st.site(j1);
  auto Fj = F(j1);
  double wj = NB_H ? st.occ(j1) : 1.0;
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the loop's own waits then count only what the loop requests
  do {
    const auto g = geom(b);
    const int jc = j1, rc = r1;
    const auto Fc = Fj;
    const double wc = wj;
    j1 = j2;
    r1 = r2;
    b = st.site(j1);
    Fj = F(j1);
    if (NB_H) wj = st.occ(j1);
    e += t + 2 * K < n ? step : 0;
    j2 = oj[e];
    r2 = orv[e];
    eval(g, Fc, wc, jc, rc);
    t += K;
  } while (t < n);
}

}  // namespace
}  // namespace a2c
