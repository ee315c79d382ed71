// Cell-list neighbor build: replaces findNeighbors (neighbors.cpp:8-113) and
// Minimizer::findLocalNeighbors (minimizer.cpp:833-1144).
//
// Set semantics (bit-exact with the oracle): j != i and
// ((dx*dx + dy*dy) + dz*dz) <= rc*rc, d = q_j - q_i in FP64, evaluated with
// contraction off so no FMA changes a borderline pair (neighbors.cpp:79-82).
// Periodic axes use d -= L*rint(d/L).  Shells: PdPdnum counts d2 < 0.75a^2,
// 0.75a^2 < d2 < 1.25a^2, else (minimizer.cpp:935-947); HH1 = H neighbors with
// d2 < 0.75a^2 (:999-1004).
//
// Passes, all on the device.  The host waits once, for the list widths after the
// count pass (the caller's positions have been read by then), and on a specimen
// with a non-periodic axis once before, for the bounding box; the passes behind the
// widths are still queued when the build returns, and whoever reads the lists from
// the host waits for the stream first:
//   k_bin     cell of each site and the cell histogram
//   k_scan    exclusive scan of the histogram (one workgroup)
//   k_place   positions as floats in cell order, with the site index, so a
//             candidate is one 16-byte load
//   k_site<false>  one wave per site: its 27 cells' candidates filtered in FP32,
//             the survivors tested in FP64; row lengths, the owned/received
//             split of each pair list, and their maxima
//   k_site<true>   the same walk keeps each hit (neighbor index and flags); the
//             wave ranks the row's hits, then the workgroup writes its 32
//             rows and their owned and received halves slot by slot
//   k_orv     the owned pairs' slots in their partners' received halves
// Rows come out sorted whatever order the cell placement used.
#pragma clang fp contract(off)

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "fe_internal.hpp"

namespace a2c {
namespace {

struct Grid {
  int nc[3];
  double lo[3], w[3];  // origin and cell width per axis
  int periodic[3];
  double box[3];
};

__device__ __forceinline__ int cell_axis(const Grid& g, double x, int c) {
  if (g.periodic[c]) x -= g.box[c] * floor(x / g.box[c]);
  int k = (int)floor((x - g.lo[c]) / g.w[c]);
  return min(max(k, 0), g.nc[c] - 1);
}

__global__ void k_bin(const double* __restrict__ X, int N, Grid g, int* __restrict__ cid,
                      int* __restrict__ ccount) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= N) return;
  int cx = cell_axis(g, X[4 * s], 0), cy = cell_axis(g, X[4 * s + 1], 1), cz = cell_axis(g, X[4 * s + 2], 2);
  int c = (cz * g.nc[1] + cy) * g.nc[0] + cx;
  cid[s] = c;
  atomicAdd(&ccount[c], 1);
}

// start[i] = sum of cnt[0..i), start[n] = the total; cursor = start[0..n).
// One workgroup: each thread scans a contiguous chunk, the chunk sums are
// scanned across the workgroup.
constexpr int SCAN_T = 1024;
__global__ __launch_bounds__(SCAN_T) void k_scan(const int* cnt, int n, int* __restrict__ start, int* cursor) {
  __shared__ int sm[SCAN_T];
  const int per = (n + SCAN_T - 1) / SCAN_T;
  const int b = min(n, (int)threadIdx.x * per), e = min(n, b + per);
  int acc = 0;
  for (int i = b; i < e; ++i) acc += cnt[i];
  sm[threadIdx.x] = acc;
  __syncthreads();
  for (int off = 1; off < SCAN_T; off <<= 1) {  // inclusive Hillis-Steele scan of the chunk sums
    const int v = threadIdx.x >= off ? sm[threadIdx.x - off] : 0;
    __syncthreads();
    sm[threadIdx.x] += v;
    __syncthreads();
  }
  int run = sm[threadIdx.x] - acc;
  for (int i = b; i < e; ++i) {  // cnt and cursor may be one array: read before writing
    const int ci = cnt[i];
    start[i] = run;
    cursor[i] = run;
    run += ci;
  }
  if (threadIdx.x == SCAN_T - 1) start[n] = sm[SCAN_T - 1];
}

// Position on one axis relative to the grid: wrapped into [0, L) or from the
// lower bound, as a float (the filter's margin covers its rounding).
__device__ __forceinline__ float grid_pos(const Grid& g, double x, int c) {
  return (float)(g.periodic[c] ? x - g.box[c] * floor(x / g.box[c]) : x - g.lo[c]);
}

// positions in cell order, the site index in .w (its bits)
__global__ void k_place(const double* __restrict__ X, int N, Grid g, const int* __restrict__ cid,
                        int* __restrict__ cursor, float4* __restrict__ qs) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= N) return;
  const int pos = atomicAdd(&cursor[cid[s]], 1);
  qs[pos] = make_float4(grid_pos(g, X[4 * s], 0), grid_pos(g, X[4 * s + 1], 1), grid_pos(g, X[4 * s + 2], 2),
                        __int_as_float(s));
}

// clears the cell histogram and the build's counters
__global__ void k_clear(int* __restrict__ a, int na, int* __restrict__ b, int nb) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < na + nb; i += gridDim.x * blockDim.x)
    (i < na ? a[i] : b[i - na]) = 0;
}

struct NbrArgs {
  const double* X;
  const float4* qs;    // cell-ordered positions
  int npd, N;
  Grid g;
  double ibox[3];
  double in0, in01;    // 1 / cells per row, 1 / cells per layer
  float fbox[3], fibox[3];  // periodic axes: L and 1 / L, else 0
  float rcf2;          // square of rc and the filter's margin
  const int* cid;
  const int* cstart;
  double rc2, sh1, sh2;
  int cap;
  int width;           // fill pass: LDS slots per row (the longest row)
  int32_t* cnt[5];     // row lengths: PdPd, PdH (Pd rows); HPd, HH, HH1 (H rows)
  int32_t* ocnt[4];    // owned entries of the four pair lists
  int32_t* rcnt[4];    // received entries
  int32_t* idx[5];     // ELL arrays (fill pass)
  int32_t* oj[4];      // owned halves (fill pass; null: no split wanted)
  int32_t* rj[4];      // received halves, species-local site indices (for k_orv)
  int32_t* pdpdnum;    // nPd*3 (fill pass)
  int32_t* maxw;       // 14 ints: width of the 5 lists, owned widths of the 4 pair lists, received
                       // widths, max total (count pass)
  int32_t* overflow;   // 1 if a site exceeds cap
  unsigned long long* totals;  // entries of the 5 lists (count pass)
};

// Ownership of the unordered pair {s, j} (global site indices) in the
// pair-once evaluation: (s < j) XOR ((s ^ j) & 1), which hands each site
// about half of every list.
__device__ __forceinline__ bool pair_owner(int s, int j) { return (s < j) != (((s ^ j) & 1) != 0); }

// d - L rint(d / L) on a periodic axis.  The quotient is formed as d (1/L):
// the two agree except within an ulp of a half-integer, where the division
// itself decides (a candidate about L/2 away, so the chosen image and the set
// stay exactly those of the division).
__device__ __forceinline__ double wrap(double d, double L, double iL) {
  const double q = d * iL;
  const double f = fabs(q - trunc(q));
  return d - L * rint(fabs(f - 0.5) < 1e-9 ? d / L : q);
}

// stencil coordinate k in 0..2 of axis ax around c: the wrapped (periodic)
// or clipped (-1: outside) cell, each distinct cell once
__device__ __forceinline__ int stencil_axis(const NbrArgs& a, int ax, int c, int k) {
  const int n = a.g.nc[ax];
  if (a.g.periodic[ax]) {
    if (n == 1) return k == 1 ? 0 : -1;  // periodic axes have 1 or >= 3 cells
    const int v = c + k - 1;
    return v < 0 ? v + n : v >= n ? v - n : v;
  }
  const int v = c + k - 1;
  return (v >= 0 && v < n) ? v : -1;
}

constexpr int NT = 64;  // rows per workgroup of k_refresh: one lane each
constexpr int CS = NT + 1;  // LDS: slot t of lane l at t * CS + l (a column and a slot row are both
                            // conflict-free)

// Build counters (list widths and totals) in SPREAD copies, a workgroup
// adding to copy blockIdx % SPREAD: tens of thousands of atomics on one
// address serialise in its L2 channel (measured: 64-thread workgroups
// spent ~0.6 ms of a 0.7 ms pass there).  The host reduces the copies.
// Layout of the context's misc buffer (bytes): SPREAD x 16 int32 (the 14
// maxima, the overflow flag in copy 0, one spare), SPREAD x 5 uint64
// (totals), the squared largest displacement, 6 bounding-box keys.
constexpr int SPREAD = 64;
constexpr size_t MISC_TOT = SPREAD * 16 * sizeof(int32_t);
constexpr size_t MISC_DMAX = MISC_TOT + SPREAD * 5 * sizeof(unsigned long long);
constexpr size_t MISC_BBOX = MISC_DMAX + sizeof(unsigned long long);
constexpr size_t MISC_BYTES = MISC_BBOX + 6 * sizeof(unsigned long long);
// The copies reduced, one lane each, to pinned memory.
__global__ __launch_bounds__(SPREAD) void k_counters(const int32_t* __restrict__ m,
                                                     const unsigned long long* __restrict__ tot,
                                                     const double* __restrict__ dmax, NbrCounters* out) {
  const int c = threadIdx.x;
#pragma unroll
  for (int k = 0; k < 14; ++k) {
    int v = m[c * 16 + k];
    for (int off = SPREAD / 2; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off));
    if (c == 0) out->max[k] = v;
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    unsigned long long v = tot[c * 5 + k];
    for (int off = SPREAD / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (c == 0) out->total[k] = v;
  }
  if (c == 0) {
    out->max[14] = m[14];
    out->max[15] = 0;
    out->d2 = *dmax;
  }
}
__device__ __forceinline__ int32_t* maxw_copy(int32_t* m) { return m + (blockIdx.x % SPREAD) * 16; }
__device__ __forceinline__ unsigned long long* tot_copy(unsigned long long* t) { return t + (blockIdx.x % SPREAD) * 5; }

// Orders a wave's own LDS writes before its reads of other lanes' words.
__device__ __forceinline__ void wave_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ int below(uint64_t mask) {  // set bits of mask under this lane
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}

// n distinct keys (16-byte aligned, padded to a multiple of four with words of
// ones): the key of rank r to out[r * RS].
constexpr int SR = 32, SW = 8, ST = 64 * SW;  // rows, waves and lanes per workgroup of k_site
constexpr int RS = SR + 1;  // LDS: slot t of row l at t * RS + l (a column and a slot row are both conflict-free)
__device__ __forceinline__ void rank_keys(const uint32_t* keys, int n, uint32_t* out, int lane) {
  for (int q = 0; q < n; q += 64) {
    const bool in = q + lane < n;
    const uint32_t mine = in ? keys[q + lane] : 0u;
    int rk = 0;
    for (int t = 0; t < n; t += 4) {
      const uint4 o = *reinterpret_cast<const uint4*>(keys + t);
      rk += (o.x < mine) + (o.y < mine) + (o.z < mine) + (o.w < mine);
    }
    if (in) out[rk * RS] = mine;
  }
}

// One wave per site, SR consecutive rows of one species per workgroup
// (Pd-row workgroups first), SR / SW sites in turn to a wave.  The site's cells
// share the wave's lanes evenly; each lane walks its cell's candidates, four
// loads in flight, in FP32 against rc plus a margin that covers the floats'
// rounding, and the survivors queue in LDS for the exact FP64 test, 64 at a time.
// Count pass (FILL = false): row lengths, owned/received counts and their
// maxima.  Fill pass: each hit's key (j << 2 | owned << 1 | first shell), Pd and
// H apart, is ranked among the row's and goes to the row's LDS column, with the
// order of the owned and received halves beside it; the workgroup then writes
// lists and halves slot by slot, SR consecutive rows per store.
// With one lane per site both passes were bound by latency at every size below
// 50,000 sites, and by the divergent loads above (count / fill pass, then the
// split, now part of the fill, and k_orv): 32,640 sites 322 / 467 / 70 / 231 us,
// now 64 / 90 / - / 12; 262,144 sites at rc + 0.2 A 805 / 1648 us, now 405 / 591.
template <bool FILL>
__global__ __launch_bounds__(ST) void k_site(NbrArgs a, int nblk_pd) {
  extern __shared__ uint32_t buf[];  // fill pass: width columns' slots, then their halves' order (bytes)
  __shared__ uint32_t queue[SW][128];
  __shared__ __align__(16) uint32_t kp[SW][FILL ? NBR_CAP : 4], kh[SW][FILL ? NBR_CAP : 4];
  __shared__ int2 cells[SW][32];
  __shared__ int counts[7][SR];  // per row: Pd and H neighbors, owned ones, HH1, the Pd shells
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int blk = xcd_block();
  const bool pdb = blk < nblk_pd;
  const int nrows = pdb ? a.npd : a.N - a.npd, soff = pdb ? 0 : a.npd;
  const int row0 = (pdb ? blk : blk - nblk_pd) * SR;
  uint8_t* const perm = reinterpret_cast<uint8_t*>(buf + (size_t)a.width * RS);
  const A2C_GLOBAL float4* __restrict__ qs = gmem(a.qs);
  const A2C_GLOBAL double4* __restrict__ X = gmem(reinterpret_cast<const double4*>(a.X));
  const A2C_GLOBAL int* __restrict__ cstart = gmem(a.cstart);
  const int kx = lane % 3, ky = (lane / 3) % 3, kz = lane / 9;  // lanes 0..26: the site's cells
  uint32_t* const que = queue[wv];
  for (int i = 0; i < SR / SW; ++i) {
    const int rl = wv * (SR / SW) + i, row = row0 + rl;
    int npn = 0, nhn = 0, op = 0, oh = 0, n1 = 0, sh0 = 0, sh1n = 0;
    if (row < nrows) {
      const int s = soff + row;
      const double4 qi = X[s];
      const float f0 = grid_pos(a.g, qi.x, 0), f1 = grid_pos(a.g, qi.y, 1), f2 = grid_pos(a.g, qi.z, 2);
      // its cells that hold sites, a power of two of lanes to each
      int start = 0, len = 0;
      {
        const int c = a.cid[s];
        const int n0 = a.g.nc[0], n01 = n0 * a.g.nc[1];
        const int cz = (int)(((double)c + 0.5) * a.in01), cyx = c - cz * n01;
        const int cy = (int)(((double)cyx + 0.5) * a.in0), cx = cyx - cy * n0;
        if (lane < 27) {
          const int xx = stencil_axis(a, 0, cx, kx), yy = stencil_axis(a, 1, cy, ky), zz = stencil_axis(a, 2, cz, kz);
          if (xx >= 0 && yy >= 0 && zz >= 0) {
            const int e = zz * n01 + yy * n0 + xx;
            start = cstart[e];
            len = cstart[e + 1] - start;
          }
        }
      }
      const uint64_t full = __ballot(len > 0);
      const int m = __popcll(full);
      const int lg = m > 1 ? 6 - (32 - __builtin_clz(m - 1)) : 6;  // log2 of the lanes per cell
      if (len > 0) cells[wv][below(full)] = make_int2(start, len);
      wave_lds();
      const int g = lane >> lg;
      const int2 mine = g < m ? cells[wv][g] : make_int2(0, 0);
      int head = 0, qn = 0;
      // exact test of the queue's first cnt (<= 64) candidates
      auto drain = [&](int cnt) {
        wave_lds();
        const bool on = lane < cnt;
        const int j = on ? (int)que[(head + lane) & 127] : s;
        const double4 qj = X[j];
        double d0 = qj.x - qi.x, d1 = qj.y - qi.y, dz = qj.z - qi.z;
        if (a.g.periodic[0]) d0 = wrap(d0, a.g.box[0], a.ibox[0]);
        if (a.g.periodic[1]) d1 = wrap(d1, a.g.box[1], a.ibox[1]);
        if (a.g.periodic[2]) dz = wrap(dz, a.g.box[2], a.ibox[2]);
        const double dd = d0 * d0 + d1 * d1 + dz * dz;
        const bool hit = on && j != s && dd <= a.rc2, jpd = j < a.npd, own = pair_owner(s, j), first = dd < a.sh1;
        const uint64_t mp = __ballot(hit && jpd), mh = __ballot(hit && !jpd), mo = __ballot(own), m1 = __ballot(first);
        if (FILL && hit) {
          const uint32_t key = ((uint32_t)j << 2) | (own ? 2u : 0u) | (first ? 1u : 0u);
          const int at = jpd ? npn + below(mp) : nhn + below(mh);
          if (at < NBR_CAP) (jpd ? kp : kh)[wv][at] = key;
        }
        npn += __popcll(mp);
        nhn += __popcll(mh);
        op += __popcll(mp & mo);
        oh += __popcll(mh & mo);
        n1 += __popcll(mh & m1);
        if (FILL) {
          sh0 += __popcll(mp & m1);
          sh1n += __popcll(__ballot(hit && jpd && dd > a.sh1 && dd < a.sh2));
        }
        head = (head + cnt) & 127;
        qn -= cnt;
        wave_lds();
      };
      const int step = 1 << lg;
      for (int e0 = lane & (step - 1); __ballot(e0 < mine.y); e0 += 4 * step) {
        float4 cq[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int e = e0 + u * step;
          cq[u] = qs[mine.x + (e < mine.y ? e : 0)];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          float d0 = cq[u].x - f0, d1 = cq[u].y - f1, dz = cq[u].z - f2;
          d0 = fmaf(-a.fbox[0], rintf(d0 * a.fibox[0]), d0);
          d1 = fmaf(-a.fbox[1], rintf(d1 * a.fibox[1]), d1);
          dz = fmaf(-a.fbox[2], rintf(dz * a.fibox[2]), dz);
          const float dd = fmaf(d0, d0, fmaf(d1, d1, dz * dz));
          const bool near = e0 + u * step < mine.y && !(dd > a.rcf2);  // NaN: left to the exact test
          const uint64_t mask = __ballot(near);
          if (near) que[(head + qn + below(mask)) & 127] = __float_as_uint(cq[u].w);
          qn += __popcll(mask);
          if (qn >= 64) drain(64);
        }
      }
      if (qn > 0) drain(qn);
      if (!FILL && lane == 0 && npn + nhn > a.cap) atomicOr(a.overflow, 1);
      if (FILL && npn + nhn <= a.width) {
        if (lane < 3 && npn + lane < NBR_CAP) kp[wv][npn + lane] = ~0u;
        if (lane < 3 && nhn + lane < NBR_CAP) kh[wv][nhn + lane] = ~0u;
        wave_lds();
        rank_keys(kp[wv], npn, buf + rl, lane);
        rank_keys(kh[wv], nhn, buf + (size_t)npn * RS + rl, lane);
        wave_lds();
        // order of the halves: owned Pd, received Pd, owned H, received H
        const int n = npn + nhn;
        int obp = 0, obh = 0, ob1 = 0;
        for (int q = 0; q < n; q += 64) {
          const int t = q + lane;
          const uint32_t key = t < n ? buf[t * RS + rl] : 0u;
          const bool own = (key & 2u) != 0, isp = t < npn;
          const uint64_t mp = __ballot(own && isp), mh = __ballot(own && !isp);
          const int bp = obp + below(mp), bh = obh + below(mh);
          if (t < n) {
            const int slot = isp ? (own ? bp : op + t - bp) : npn + (own ? bh : oh + t - npn - bh);
            perm[slot * RS + rl] = (uint8_t)t;
          }
          obp += __popcll(mp);
          obh += __popcll(mh);
          if (!pdb) {  // HH1, in order
            const uint64_t m1 = __ballot(t < n && !isp && (key & 1u));
            if (t < n && !isp && (key & 1u))
              a.idx[4][(size_t)(ob1 + below(m1)) * nrows + row] = (int)(key >> 2) - a.npd;
            ob1 += __popcll(m1);
          }
        }
      }
    }
    if (lane == 0) {
      counts[0][rl] = npn; counts[1][rl] = nhn; counts[2][rl] = op; counts[3][rl] = oh; counts[4][rl] = n1;
      counts[5][rl] = sh0; counts[6][rl] = sh1n;
    }
  }
  __syncthreads();
  const int rl = tid & (SR - 1), row = row0 + rl;
  const int npn = counts[0][rl], nhn = counts[1][rl], op = counts[2][rl], oh = counts[3][rl], n1 = counts[4][rl];
  const int lp = pdb ? 0 : 2, lh = pdb ? 1 : 3;
  const int p = row_of_site(row, nrows);
  if (FILL && row < nrows && npn + nhn <= a.width) {
    const int n = npn + nhn;
    const bool split = a.oj[lp] != nullptr;
    for (int t = tid / SR; t < n; t += ST / SR) {
      const int j = (int)(buf[t * RS + rl] >> 2);
      if (t < npn) a.idx[lp][(size_t)t * nrows + row] = j;
      else a.idx[lh][(size_t)(t - npn) * nrows + row] = j - a.npd;
      if (!split) continue;
      const int k = (int)(buf[perm[t * RS + rl] * RS + rl] >> 2);
      if (t < op) a.oj[lp][(size_t)t * nrows + p] = row_of_site(k, a.npd);
      else if (t < npn) a.rj[lp][(size_t)(t - op) * nrows + p] = k;
      else if (t < npn + oh) a.oj[lh][(size_t)(t - npn) * nrows + p] = row_of_site(k - a.npd, a.N - a.npd);
      else a.rj[lh][(size_t)(t - npn - oh) * nrows + p] = k - a.npd;
    }
  }
  if (tid >= 64) return;
  const bool live = tid < SR && row < nrows;
  if (!FILL) {
    if (live) {
      a.cnt[lp][row] = npn;
      a.cnt[lh][row] = nhn;
      a.ocnt[lp][p] = op;
      a.rcnt[lp][p] = npn - op;
      a.ocnt[lh][p] = oh;
      a.rcnt[lh][p] = nhn - oh;
      if (!pdb) a.cnt[4][row] = n1;
    }
    // maxima over the workgroup, then one atomic per quantity (rows past the end count 0)
    int v[14] = {0};
    v[lp] = npn; v[lh] = nhn; v[4] = pdb ? 0 : n1;
    v[5 + lp] = op; v[5 + lh] = oh; v[9 + lp] = npn - op; v[9 + lh] = nhn - oh; v[13] = npn + nhn;
#pragma unroll
    for (int k = 0; k < 14; ++k) {
      int m = v[k];
      for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off));
      v[k] = m;
    }
    if (lane == 0) {
      int32_t* mw = maxw_copy(a.maxw);
#pragma unroll
      for (int k = 0; k < 14; ++k)
        if (v[k]) atomicMax(&mw[k], v[k]);
    }
    // totals of the five lists: sums over the workgroup, one atomic each
    unsigned long long tp = live ? npn : 0, th = live ? nhn : 0, t1 = live && !pdb ? n1 : 0;
    for (int off = 32; off > 0; off >>= 1) {
      tp += __shfl_xor(tp, off);
      th += __shfl_xor(th, off);
      t1 += __shfl_xor(t1, off);
    }
    if (lane == 0) {
      unsigned long long* tt = tot_copy(a.totals);
      atomicAdd(&tt[lp], tp);
      atomicAdd(&tt[lh], th);
      if (!pdb) atomicAdd(&tt[4], t1);
    }
    return;
  }
  if (live && pdb) {
    a.pdpdnum[3 * (size_t)row] = counts[5][rl];
    a.pdpdnum[3 * (size_t)row + 1] = counts[6][rl];
    a.pdpdnum[3 * (size_t)row + 2] = npn - counts[5][rl] - counts[6][rl];
  }
}

// For every owned entry (list blockIdx.z; a row's entries dealt to ORV_Y threads):
// the received slot of its row in the partner row, found by binary search of
// the partner's received half (sorted site indices, in rbuf until the first
// evaluation; if absent, which the symmetric lists never produce, a slot past
// the received half that nothing reads: the owner passes store every share
// without a test).  Neighboring rows' entries of one slot probe neighboring rows.
constexpr int ORV_Y = 16;
struct OrvArgs {
  Ell L[4];
  int spare[4];   // that slot, per partner list
  int32_t* maxw;  // after a refresh: the longest total row (Pd rows: PdPd + PdH, H rows: HPd + HH) goes to maxw[13]
};
__global__ void k_orv(OrvArgs a) {
  const int w = blockIdx.z;
  const Ell& L = a.L[w];
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (a.maxw && blockIdx.y == 0 && w % 2 == 0) {
    int m = p < L.rows ? L.cnt[p] + a.L[w + 1].cnt[p] : 0;
    for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0 && m) atomicMax(&maxw_copy(a.maxw)[13], m);
  }
  if (p >= L.rows) return;
  const int pw = w == 1 ? 2 : w == 2 ? 1 : w;  // PdPd, PdH <-> HPd, HH
  const Ell& P = a.L[pw];
  const int r = site_of_row(p, L.rows), n = L.ocnt[p];
  for (int t = blockIdx.y; t < n; t += ORV_Y) {
    const size_t e = (size_t)t * L.rows + p;
    const int j = L.oj[e];
    const A2C_GLOBAL int32_t* rj = gmem(reinterpret_cast<const int32_t*>(P.rbuf)) + j;
    int lo = 0, hi = P.rcnt[j];  // the slot is in [lo, hi) if the row holds r
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (rj[(size_t)mid * P.rows] <= r) lo = mid;
      else hi = mid;
    }
    L.orv[e] = lo < hi && rj[(size_t)lo * P.rows] == r ? lo : a.spare[pw];
  }
}

// Bounding box of the positions (non-periodic axes): per block, then one
// atomic per block and quantity on the ordered-integer image of the double.
__device__ __forceinline__ unsigned long long dkey(double x) {  // monotone map double -> uint64
  const unsigned long long u = (unsigned long long)__double_as_longlong(x);
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__global__ __launch_bounds__(256) void k_bbox(const double* __restrict__ X, int N, unsigned long long* out) {
  __shared__ unsigned long long red[6][256];
  unsigned long long lo[3] = {~0ull, ~0ull, ~0ull}, hi[3] = {0ull, 0ull, 0ull};
  for (int s = blockIdx.x * 256 + threadIdx.x; s < N; s += gridDim.x * 256)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const unsigned long long k = dkey(X[4 * (size_t)s + c]);
      lo[c] = min(lo[c], k);
      hi[c] = max(hi[c], k);
    }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    red[c][threadIdx.x] = lo[c];
    red[3 + c][threadIdx.x] = hi[c];
  }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        red[c][threadIdx.x] = min(red[c][threadIdx.x], red[c][threadIdx.x + w]);
        red[3 + c][threadIdx.x] = max(red[3 + c][threadIdx.x], red[3 + c][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 3) atomicMin(&out[threadIdx.x], red[threadIdx.x][0]);
  else if (threadIdx.x < 6) atomicMax(&out[threadIdx.x], red[threadIdx.x][0]);
}
double dkey_inv(unsigned long long k) {
  const unsigned long long u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
  double x;
  std::memcpy(&x, &u, 8);
  return x;
}

// ---------------------------------------------------------------- skin lists
// Largest squared displacement of any site from its position at the skin
// build (minimum image on periodic axes), as the bit pattern of a
// non-negative double (ordered like the value).
__global__ __launch_bounds__(256) void k_maxdisp(const double* __restrict__ X, const double* __restrict__ X0, int N,
                                                 Grid g, unsigned long long* out) {
  __shared__ double red[256];
  double m = 0.0;
  for (int s = blockIdx.x * 256 + threadIdx.x; s < N; s += gridDim.x * 256) {
    double d2 = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double d = X[4 * (size_t)s + c] - X0[4 * (size_t)s + c];
      if (g.periodic[c]) d -= g.box[c] * rint(d / g.box[c]);
      d2 += d * d;
    }
    m = fmax(m, d2);
  }
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicMax(out, (unsigned long long)__double_as_longlong(red[0]));
}

struct RefreshArgs {
  const double* X;
  int npd, N;
  Grid g;
  double ibox[3];
  double rc2, sh1, sh2;
  Ell sup[4];          // skin lists: PdPd, PdH (Pd rows), HPd, HH (H rows)
  Ell out[5];          // lists at rc (idx, cnt; pair lists also ocnt, rcnt, oj, and the received half in rbuf)
  int32_t* pdpdnum;
  int32_t* maxw;       // 14 ints as in the count pass
  unsigned long long* totals;
  const unsigned long long* dmax;  // squared largest displacement (a double's bits), 0 after a skin build
};

__device__ __forceinline__ int wave_max(int v) {
  for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off));
  return v;
}

// One lane per row of one list (one wave per workgroup; the workgroups of
// PdPd, PdH, HPd and HH rows in that order): the row's skin-list entries
// still within rc, in the skin list's (sorted) order, into the list at rc
// with its owned/received split, and the Pd shell counts (PdPd) or HH1
// (HH) -- the count and fill passes' results for the same positions,
// without the cell walk.  An entry whose distance at the skin build (kept as
// a float beside it) is further than 2 delta + 1e-6 A from rc and from the
// shell radii, delta the largest displacement since then, is decided by that
// distance alone: no site pair moved closer or apart by more than 2 delta,
// and the float carries 3e-7 A of rounding.  The others are tested with the
// current FP64 positions exactly as the cell walk tests them.  Kept
// entries are staged in the lane's LDS column (neighbor << 2 | owned << 1 |
// first shell), then each output array is written slot by slot, 64
// consecutive rows per store.
// 262,144 sites, rebuilt in place: 176 us with one entry's positions at a time, 124
// with a batch's (the lists' own bytes take 70); the reverse slots 73 us from the
// received halves, where per-entry fates and twins took 157 us in four launches.
__global__ __launch_bounds__(NT) void k_refresh(RefreshArgs a, int4 blk0) {
  extern __shared__ uint32_t col[];
  const int b = blockIdx.x;
  const int w = b < blk0.y ? 0 : (b < blk0.z ? 1 : (b < blk0.w ? 2 : 3));  // the list of this workgroup
  const int b0 = w == 0 ? 0 : (w == 1 ? blk0.y : (w == 2 ? blk0.z : blk0.w));
  const bool pdr = w < 2;                                 // Pd rows
  const int nrows = pdr ? a.npd : a.N - a.npd;
  const int lane = (int)threadIdx.x;
  const int row = (b - b0) * NT + lane;
  const int prow = row_of_site(row, nrows);              // of the split lists
  const int jrows = (w == 0 || w == 2) ? a.npd : a.N - a.npd;
  const bool live = row < nrows;
  const int s = (pdr ? 0 : a.npd) + (live ? row : 0);
  const int joff = (w == 0 || w == 2) ? 0 : a.npd;       // neighbors: Pd for PdPd and HPd
  const bool shells = w == 0, first = w == 3;             // PdPdnum / HH1
  const A2C_GLOBAL double4* __restrict__ X = gmem(reinterpret_cast<const double4*>(a.X));
  const double band = 2.0 * sqrt(__longlong_as_double((long long)*a.dmax)) + 1e-6;
  const double r1 = sqrt(a.sh1), r2 = sqrt(a.sh2), rc = sqrt(a.rc2);
  const double4 qi = X[s];
  const Ell S = a.sup[w];
  const Ell L = a.out[w];
  const A2C_GLOBAL int32_t* __restrict__ sidx = gmem(S.idx);
  const A2C_GLOBAL float* __restrict__ sdist = gmem(reinterpret_cast<const float*>(S.oj));
  const size_t srows = S.rows, orows = L.rows;
  const int n = live ? gmem(S.cnt)[row] : 0;
  int nk = 0, no = 0, nr = 0, nf = 0, sh0 = 0, sh1n = 0;
  // Entries in batches of B: the next batch's indices and distances are
  // requested before this one is decided, and where some lane needs positions, all
  // of the batch's are requested together.
  constexpr int B = 8;
  const int nw = wave_max(n);
  int jb[B], jn[B];
  float db[B], dn[B];
  auto load = [&](int t0, int (&jv)[B], float (&dv)[B]) {
#pragma unroll
    for (int u = 0; u < B; ++u) {  // past the row's end its last entry again
      const size_t se = (size_t)max(min(t0 + u, n - 1), 0) * srows + (live ? row : 0);
      jv[u] = sidx[se];
      dv[u] = sdist[se];
    }
  };
  if (nw > 0) load(0, jn, dn);
  for (int t0 = 0; t0 < nw; t0 += B) {
#pragma unroll
    for (int u = 0; u < B; ++u) {
      jb[u] = jn[u];
      db[u] = dn[u];
    }
    load(t0 + B, jn, dn);
    bool near[B], keep[B], some = false;
    int cls[B];  // shell class: 0 below r1, 1 between, 2 beyond
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const double df = (double)db[u];
      const bool near_rc = fabs(df - rc) <= band;
      const bool near_sh = (shells || first) && (fabs(df - r1) <= band || (shells && fabs(df - r2) <= band));
      near[u] = t0 + u < n && (near_rc || near_sh);
      some |= near[u];
      keep[u] = t0 + u < n && df < rc;
      cls[u] = df < r1 ? 0 : (df < r2 ? 1 : 2);
    }
    if (__ballot(some)) {
      double4 q[B];
#pragma unroll
      for (int u = 0; u < B; ++u) q[u] = X[near[u] ? joff + jb[u] : s];
#pragma unroll
      for (int u = 0; u < B; ++u) {
        double d0 = q[u].x - qi.x, d1 = q[u].y - qi.y, dz = q[u].z - qi.z;
        if (a.g.periodic[0]) d0 = wrap(d0, a.g.box[0], a.ibox[0]);
        if (a.g.periodic[1]) d1 = wrap(d1, a.g.box[1], a.ibox[1]);
        if (a.g.periodic[2]) dz = wrap(dz, a.g.box[2], a.ibox[2]);
        const double d2 = d0 * d0 + d1 * d1 + dz * dz;
        if (near[u]) {
          keep[u] = d2 <= a.rc2;
          cls[u] = d2 < a.sh1 ? 0 : ((d2 > a.sh1 && d2 < a.sh2) ? 1 : 2);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      if (!keep[u]) continue;
      const bool owned = pair_owner(s, joff + jb[u]);
      owned ? ++no : ++nr;
      if (shells) {
        if (cls[u] == 0) ++sh0;
        else if (cls[u] == 1) ++sh1n;
      }
      const bool f1 = first && cls[u] == 0;
      nf += f1;
      col[nk * CS + lane] = ((uint32_t)jb[u] << 2) | (owned ? 2u : 0u) | (f1 ? 1u : 0u);
      ++nk;
    }
  }
  // the wave's longest row, halves and HH1 row: slot loops every lane joins
  int mk = nk, mo = no, mr = nr, mf = nf;
  for (int off = 32; off > 0; off >>= 1) {
    mk = max(mk, __shfl_xor(mk, off));
    mo = max(mo, __shfl_xor(mo, off));
    mr = max(mr, __shfl_xor(mr, off));
    mf = max(mf, __shfl_xor(mf, off));
  }
  A2C_GLOBAL int32_t* __restrict__ oidx = gmem(L.idx);
  for (int u = 0; u < mk; ++u)
    if (u < nk) oidx[(size_t)u * orows + row] = (int)(col[u * CS + lane] >> 2);
  A2C_GLOBAL int32_t* __restrict__ ooj = gmem(L.oj);
  for (int u = 0, q = 0; u < mo; ++u) {
    if (u >= no) continue;
    while (!(col[q * CS + lane] & 2u)) ++q;
    ooj[(size_t)u * orows + prow] = row_of_site((int)(col[q * CS + lane] >> 2), jrows);
    ++q;
  }
  A2C_GLOBAL int32_t* __restrict__ orj = gmem(reinterpret_cast<int32_t*>(L.rbuf));
  for (int u = 0, q = 0; u < mr; ++u) {
    if (u >= nr) continue;
    while (col[q * CS + lane] & 2u) ++q;
    orj[(size_t)u * orows + prow] = (int)(col[q * CS + lane] >> 2);
    ++q;
  }
  if (first) {
    A2C_GLOBAL int32_t* __restrict__ h1 = gmem(a.out[4].idx);
    const size_t rows4 = a.out[4].rows;
    for (int u = 0, q = 0; u < mf; ++u) {
      if (u >= nf) continue;
      while (!(col[q * CS + lane] & 1u)) ++q;
      h1[(size_t)u * rows4 + row] = (int)(col[q * CS + lane] >> 2);
      ++q;
    }
  }
  if (live) {
    gmem(L.cnt)[row] = nk;
    gmem(L.ocnt)[prow] = no;
    gmem(L.rcnt)[prow] = nr;
    if (first) gmem(a.out[4].cnt)[row] = nf;
    if (shells) {
      A2C_GLOBAL int32_t* pn = gmem(a.pdpdnum);
      pn[3 * (size_t)row] = sh0;
      pn[3 * (size_t)row + 1] = sh1n;
      pn[3 * (size_t)row + 2] = nk - sh0 - sh1n;
    }
  }
  // maxima (row length, owned and received halves, HH1) and totals of the list
  int v[4] = {nk, no, nr, nf};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    int m = v[k];
    for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off));
    v[k] = m;
  }
  unsigned long long tk = nk, tf = nf;
  for (int off = 32; off > 0; off >>= 1) {
    tk += __shfl_xor(tk, off);
    tf += __shfl_xor(tf, off);
  }
  if (lane == 0) {
    int32_t* mw = maxw_copy(a.maxw);
    unsigned long long* tt = tot_copy(a.totals);
    if (v[0]) atomicMax(&mw[w], v[0]);
    if (v[1]) atomicMax(&mw[5 + w], v[1]);
    if (v[2]) atomicMax(&mw[9 + w], v[2]);
    if (first && v[3]) atomicMax(&mw[4], v[3]);
    atomicAdd(&tt[w], tk);
    if (first) atomicAdd(&tt[4], tf);
  }
}

// Skin build: the FP64 distance of every skin entry (as the cell walk
// computes it), rounded to a float, into the skin list's oj.
__global__ void k_sdist(Ell L, const double* __restrict__ X, int s_off, int j_off, Grid g, double ix, double iy,
                        double iz) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int t = blockIdx.y;
  if (r >= L.rows || t >= L.cnt[r]) return;
  const size_t e = (size_t)t * L.rows + r;
  const A2C_GLOBAL double4* __restrict__ Q = gmem(reinterpret_cast<const double4*>(X));
  const double4 qi = Q[s_off + r], qj = Q[j_off + L.idx[e]];
  double d0 = qj.x - qi.x, d1 = qj.y - qi.y, dz = qj.z - qi.z;
  if (g.periodic[0]) d0 = wrap(d0, g.box[0], ix);
  if (g.periodic[1]) d1 = wrap(d1, g.box[1], iy);
  if (g.periodic[2]) dz = wrap(dz, g.box[2], iz);
  reinterpret_cast<float*>(L.oj)[e] = (float)sqrt(d0 * d0 + d1 * d1 + dz * dz);
}

}  // namespace

namespace {

// The counters of a build on the host: c->nb_host, pinned, written by k_counters
// and valid after a synchronisation.
void read_counters(const a2c_fe_ctx* c, int hm[16], unsigned long long ht[5]) {
  std::memcpy(hm, c->nb_host->max, sizeof(c->nb_host->max));
  for (int k = 0; k < 5; ++k) ht[k] = c->nb_host->total[k];
}
int launch_counters(a2c_fe_ctx* c) {
  const char* m = reinterpret_cast<const char*>(c->nb_misc);
  hipLaunchKernelGGL(k_counters, dim3(1), dim3(SPREAD), 0, c->stream, c->nb_misc,
                     reinterpret_cast<const unsigned long long*>(m + MISC_TOT),
                     reinterpret_cast<const double*>(m + MISC_DMAX), c->nb_host);
  A2C_HIP(c, hipGetLastError());
  return A2C_OK;
}
int nbr_counters(a2c_fe_ctx* c) {  // the buffers of a build's counters
  if (!c->nb_misc) A2C_HIP(c, dmalloc(&c->nb_misc, MISC_BYTES));
  if (!c->nb_host) A2C_HIP(c, hmalloc(&c->nb_host, sizeof(NbrCounters)));
  return A2C_OK;
}

// Device buffers of one set of five lists for rows of npd / nh sites: row
// counts always; ELL arrays, owned halves and received-share buffers for
// list widths w[0..4], owned widths ow[0..3] and received widths rw[0..3]
// (grow-only, with slack so small width changes reuse the arrays).
int size_lists(a2c_fe_ctx* c, Ell* L5, const int* w, const int* ow, const int* rw) {
  const int npd = c->desc.n_pd, nh = c->desc.n_h;
  for (int k = 0; k < 5; ++k) {
    Ell& L = L5[k];
    L.rows = (k < 2) ? npd : nh;
    const int64_t rows = std::max(L.rows, 1);
    if (!L.cnt) A2C_HIP(c, dmalloc(&L.cnt, sizeof(int32_t) * rows));
    if (k < 4 && !L.ocnt) {
      A2C_HIP(c, dmalloc(&L.ocnt, sizeof(int32_t) * rows));
      A2C_HIP(c, dmalloc(&L.rcnt, sizeof(int32_t) * rows));
    }
    if (!w) continue;
    const int64_t n = (int64_t)std::max(w[k], 1) * rows;
    if (n > L.cap) {
      (void)dfree(L.idx);
      L.idx = nullptr;
      L.cap = (int64_t)(std::max(w[k], 1) + 4) * rows;
      A2C_HIP(c, dmalloc(&L.idx, sizeof(int32_t) * L.cap));
    }
    if (k == 4 || !ow) continue;
    const int64_t on = (int64_t)std::max(ow[k], 1) * rows;
    const int64_t rn = (int64_t)(std::max(rw[k], 1) + 1) * rows;  // one slot to spare (k_orv)
    const int64_t bn = 32 * rn;
    if (on > L.ocap) {
      (void)dfree(L.oj); (void)dfree(L.orv);
      L.oj = L.orv = nullptr;
      L.ocap = on + 4 * rows;
      A2C_HIP(c, dmalloc(&L.oj, sizeof(int32_t) * L.ocap));
      A2C_HIP(c, dmalloc(&L.orv, sizeof(int32_t) * L.ocap));
    }
    if (bn > L.bcap) {
      (void)dfree(L.rbuf);
      L.rbuf = nullptr;
      L.bcap = bn + 32 * 4 * rows;
      A2C_HIP(c, dmalloc(&L.rbuf, L.bcap));
    }
  }
  return A2C_OK;
}

// Reverse slots of the four pair lists (after the fill pass or a refresh);
// spare[w]: an allocated slot past list w's received halves.
int reverse_slots(a2c_fe_ctx* c, const Ell* L5, const int* spare, int32_t* maxw) {
  OrvArgs a;
  a.maxw = maxw;
  int rows = 0;
  for (int w = 0; w < 4; ++w) {
    a.L[w] = L5[w];
    a.spare[w] = spare[w];
    rows = std::max(rows, L5[w].rows);
  }
  if (rows == 0) return A2C_OK;
  hipLaunchKernelGGL(k_orv, dim3((rows + 255) / 256, ORV_Y, 4), dim3(256), 0, c->stream, a);
  A2C_HIP(c, hipGetLastError());
  return A2C_OK;
}

Grid box_grid(a2c_fe_ctx* c) {
  Grid g{};
  for (int ax = 0; ax < 3; ++ax) {
    g.periodic[ax] = c->desc.periodic[ax];
    g.box[ax] = c->desc.box[ax];
  }
  return g;
}

// The cell walk: lists of radius rc from the positions c->dX into L5 (the
// context's lists, or its skin lists).  halves: also the owned/received
// split and the reverse slots.  hm: widths (as the count pass's maxima),
// ht: totals.
int walk_cells(a2c_fe_ctx* c, double rc, Ell* L5, bool halves, int hm[16], unsigned long long ht[5]) {
  const int N = c->N, npd = c->desc.n_pd, nh = c->desc.n_h;
  const int TB = 256;
  // scratch (grow-only)
  if (!c->nb_cid) {
    A2C_HIP(c, dmalloc(&c->nb_cid, sizeof(int) * std::max(N, 1)));
    A2C_HIP(c, dmalloc(&c->nb_order, sizeof(float4) * std::max(N, 1)));  // cell-ordered positions
  }
  if (int rc2 = nbr_counters(c)) return rc2;
  int* misc = c->nb_misc;
  unsigned long long* totals = reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(misc) + MISC_TOT);
  unsigned long long* bbox = reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(misc) + MISC_BBOX);
  Grid g = box_grid(c);
  bool need_bbox = false;
  for (int ax = 0; ax < 3; ++ax) need_bbox |= !c->desc.periodic[ax];
  double lo3[3] = {0, 0, 0}, hi3[3] = {1, 1, 1};
  if (need_bbox && N > 0) {
    unsigned long long init[6] = {~0ull, ~0ull, ~0ull, 0ull, 0ull, 0ull};
    A2C_HIP(c, hipMemcpyAsync(bbox, init, sizeof(init), hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(k_bbox, dim3(std::min((N + TB - 1) / TB, 256)), dim3(TB), 0, c->stream, c->dX, N, bbox);
    A2C_HIP(c, hipGetLastError());
    unsigned long long hb[6];
    A2C_HIP(c, hipMemcpyAsync(hb, bbox, sizeof(hb), hipMemcpyDeviceToHost, c->stream));
    A2C_HIP(c, hipStreamSynchronize(c->stream));
    for (int ax = 0; ax < 3; ++ax) {
      lo3[ax] = dkey_inv(hb[ax]);
      hi3[ax] = dkey_inv(hb[3 + ax]);
    }
  }
  for (int ax = 0; ax < 3; ++ax) {
    double lo = 0.0, hi = 1.0;
    if (g.periodic[ax]) {
      lo = 0.0; hi = g.box[ax];
    } else if (N > 0) {
      lo = lo3[ax]; hi = hi3[ax];
    }
    int nc = std::max(1, (int)std::floor((hi - lo) / rc));
    if (g.periodic[ax] && nc < 3) nc = 1;
    g.nc[ax] = nc;
    g.lo[ax] = lo;
    g.w[ax] = (hi - lo) / nc;
    if (!(g.w[ax] > 0)) g.w[ax] = 1.0;
  }
  const long long ncell = (long long)g.nc[0] * g.nc[1] * g.nc[2];
  if (ncell > (1LL << 28)) return set_err(c, A2C_EINVAL, "neighbor grid too large");
  if (ncell + 1 > c->nb_cap_cells) {
    (void)dfree(c->nb_cc);
    (void)dfree(c->nb_cursor);
    c->nb_cc = c->nb_cursor = nullptr;
    A2C_HIP(c, dmalloc(&c->nb_cc, sizeof(int) * (ncell + 1)));
    A2C_HIP(c, dmalloc(&c->nb_cursor, sizeof(int) * (ncell + 1)));
    c->nb_cap_cells = ncell + 1;
  }
  int *dcid = c->nb_cid, *dcc = c->nb_cc, *dcursor = c->nb_cursor;
  float4* qs = reinterpret_cast<float4*>(c->nb_order);
  {
    const int nm = (int)(MISC_BBOX / sizeof(int)), n = (int)ncell + 1 + nm;
    hipLaunchKernelGGL(k_clear, dim3(std::min((n + TB - 1) / TB, 1024)), dim3(TB), 0, c->stream, dcursor,
                       (int)ncell + 1, misc, nm);
    A2C_HIP(c, hipGetLastError());
  }
  if (N > 0) {
    hipLaunchKernelGGL(k_bin, dim3((N + TB - 1) / TB), dim3(TB), 0, c->stream, c->dX, N, g, dcid, dcursor);
    A2C_HIP(c, hipGetLastError());
  }
  hipLaunchKernelGGL(k_scan, dim3(1), dim3(SCAN_T), 0, c->stream, dcursor, (int)ncell, dcc, dcursor);
  A2C_HIP(c, hipGetLastError());
  if (N > 0) {
    hipLaunchKernelGGL(k_place, dim3((N + TB - 1) / TB), dim3(TB), 0, c->stream, c->dX, N, g, dcid, dcursor, qs);
    A2C_HIP(c, hipGetLastError());
  }
  if (int rc2 = size_lists(c, L5, nullptr, nullptr, nullptr)) return rc2;  // row counts
  NbrArgs a{};
  a.X = c->dX; a.qs = qs; a.npd = npd; a.N = N; a.g = g; a.cid = dcid; a.cstart = dcc;
  for (int ax = 0; ax < 3; ++ax) a.ibox[ax] = g.box[ax] > 0.0 ? 1.0 / g.box[ax] : 0.0;
  // the filter's margin: the floats' rounding over the grid's extent, with room to spare
  double extent = 0.0;
  for (int ax = 0; ax < 3; ++ax) {
    extent = std::max(extent, g.w[ax] * g.nc[ax]);
    a.fbox[ax] = g.periodic[ax] ? (float)g.box[ax] : 0.0f;
    a.fibox[ax] = g.periodic[ax] ? (float)a.ibox[ax] : 0.0f;
  }
  const double rcf = rc + 1e-4 + extent * 0x1p-20;
  a.rcf2 = (float)(rcf * rcf);
  a.in0 = 1.0 / g.nc[0];
  a.in01 = 1.0 / ((double)g.nc[0] * g.nc[1]);
  a.rc2 = rc * rc;
  a.sh1 = c->desc.a_pd * c->desc.a_pd * 0.75;
  a.sh2 = c->desc.a_pd * c->desc.a_pd * 1.25;
  a.cap = std::min(c->desc.max_neighbors > 0 ? c->desc.max_neighbors : NBR_CAP, NBR_CAP);
  for (int w = 0; w < 5; ++w) a.cnt[w] = L5[w].cnt;
  for (int w = 0; w < 4; ++w) { a.ocnt[w] = L5[w].ocnt; a.rcnt[w] = L5[w].rcnt; }
  a.maxw = misc;
  a.overflow = misc + 14;
  a.totals = totals;
  const int nblk_pd = (npd + SR - 1) / SR, nblk_h = (nh + SR - 1) / SR;
  if (nblk_pd + nblk_h > 0) {
    hipLaunchKernelGGL(k_site<false>, dim3(nblk_pd + nblk_h), dim3(ST), 0, c->stream, a, nblk_pd);
    A2C_HIP(c, hipGetLastError());
  }
  if (int rc2 = launch_counters(c)) return rc2;
  A2C_HIP(c, hipStreamSynchronize(c->stream));
  read_counters(c, hm, ht);
  if (hm[14]) return A2C_ENBR_OVERFLOW;
  if (int rc2 = size_lists(c, L5, hm, halves ? hm + 5 : nullptr, hm + 9)) return rc2;
  for (int w = 0; w < 5; ++w) {
    a.idx[w] = L5[w].idx;
    L5[w].width = hm[w];
    if (w < 4) {
      a.oj[w] = halves ? L5[w].oj : nullptr;
      a.rj[w] = halves ? reinterpret_cast<int32_t*>(L5[w].rbuf) : nullptr;
      L5[w].owidth = hm[5 + w];
      L5[w].rwidth = hm[9 + w];
    }
  }
  if (!c->dpdpdnum) A2C_HIP(c, dmalloc(&c->dpdpdnum, sizeof(int32_t) * 3 * std::max(npd, 1)));
  a.pdpdnum = c->dpdpdnum;
  a.width = std::max(hm[13], 1);
  if (nblk_pd + nblk_h > 0) {
    hipLaunchKernelGGL(k_site<true>, dim3(nblk_pd + nblk_h), dim3(ST), (sizeof(uint32_t) + 1) * RS * (size_t)a.width,
                       c->stream, a, nblk_pd);
    A2C_HIP(c, hipGetLastError());
  }
  if (halves)
    if (int rc2 = reverse_slots(c, L5, hm + 9, nullptr)) return rc2;
  return A2C_OK;
}

// Distance of every skin entry at the skin build, as a float, in oj.
int size_skin_extras(a2c_fe_ctx* c) {
  for (int k = 0; k < 4; ++k) {
    Ell& S = c->nb_sup[k];
    const int64_t n = (int64_t)std::max(S.width, 1) * std::max(S.rows, 1);
    if (n > S.ocap) {
      (void)dfree(S.oj);
      S.oj = nullptr;
      S.ocap = n + 4 * (int64_t)std::max(S.rows, 1);
      A2C_HIP(c, dmalloc(&S.oj, sizeof(float) * S.ocap));
    }
  }
  const Grid g = box_grid(c);
  double ib[3];
  for (int ax = 0; ax < 3; ++ax) ib[ax] = g.box[ax] > 0.0 ? 1.0 / g.box[ax] : 0.0;
  static const int s_sp[4] = {0, 0, 1, 1}, j_sp[4] = {0, 1, 0, 1};  // species of rows / of neighbors
  for (int k = 0; k < 4; ++k) {
    const Ell& S = c->nb_sup[k];
    if (S.rows == 0 || S.width == 0) continue;
    hipLaunchKernelGGL(k_sdist, dim3((S.rows + 255) / 256, S.width), dim3(256), 0, c->stream, S, c->dX,
                       s_sp[k] * c->desc.n_pd, j_sp[k] * c->desc.n_pd, g, ib[0], ib[1], ib[2]);
    A2C_HIP(c, hipGetLastError());
  }
  return A2C_OK;
}

// The context's lists at rc filtered from its skin lists, and (check) the
// largest displacement since the skin build, in one round trip: the caller
// keeps the result only if that displacement is under skin/2.
int refresh(a2c_fe_ctx* c, bool check, int hm[16], unsigned long long ht[5], double* maxd) {
  const int N = c->N, npd = c->desc.n_pd, nh = c->desc.n_h;
  // every list at rc fits in the capacity of its skin list
  int w[5], ow[4], rw[4];
  for (int k = 0; k < 5; ++k) w[k] = c->nb_sup[k < 4 ? k : 3].width;
  for (int k = 0; k < 4; ++k) ow[k] = rw[k] = c->nb_sup[k].width;
  if (int rc = size_lists(c, c->ell, w, ow, rw)) return rc;
  int* misc = c->nb_misc;
  unsigned long long* totals = reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(misc) + MISC_TOT);
  unsigned long long* dmax = reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(misc) + MISC_DMAX);
  hipLaunchKernelGGL(k_clear, dim3(8), dim3(256), 0, c->stream, misc, (int)(MISC_BBOX / sizeof(int)), misc, 0);
  A2C_HIP(c, hipGetLastError());
  if (!c->dpdpdnum) A2C_HIP(c, dmalloc(&c->dpdpdnum, sizeof(int32_t) * 3 * std::max(npd, 1)));
  const Grid g = box_grid(c);
  if (check && N > 0) {
    hipLaunchKernelGGL(k_maxdisp, dim3(std::min((N + 255) / 256, 256)), dim3(256), 0, c->stream, c->dX,
                       c->nb_sup_q, N, g, dmax);
    A2C_HIP(c, hipGetLastError());
  }
  RefreshArgs a{};
  a.X = c->dX;
  a.npd = npd;
  a.N = N;
  a.g = g;
  for (int ax = 0; ax < 3; ++ax) a.ibox[ax] = g.box[ax] > 0.0 ? 1.0 / g.box[ax] : 0.0;
  a.rc2 = c->desc.rc * c->desc.rc;
  a.sh1 = c->desc.a_pd * c->desc.a_pd * 0.75;
  a.sh2 = c->desc.a_pd * c->desc.a_pd * 1.25;
  for (int k = 0; k < 4; ++k) a.sup[k] = c->nb_sup[k];
  for (int k = 0; k < 5; ++k) a.out[k] = c->ell[k];
  a.pdpdnum = c->dpdpdnum;
  a.maxw = misc;
  a.totals = totals;
  a.dmax = dmax;
  const int bp = (npd + NT - 1) / NT, bh = (nh + NT - 1) / NT;  // workgroups per list of Pd / H rows
  const int4 blk0 = make_int4(0, bp, 2 * bp, 2 * bp + bh);     // first workgroup of each list
  int wmax = 1;  // LDS column of a lane: the longest skin row of any list
  for (int k = 0; k < 4; ++k) wmax = std::max(wmax, c->nb_sup[k].width);
  if (bp + bh > 0) {
    hipLaunchKernelGGL(k_refresh, dim3(2 * (bp + bh)), dim3(NT), sizeof(uint32_t) * CS * wmax, c->stream, a, blk0);
    A2C_HIP(c, hipGetLastError());
  }
  if (int rc = reverse_slots(c, c->ell, rw, misc)) return rc;  // rw + 1 slots are allocated
  if (int rc = launch_counters(c)) return rc;
  A2C_HIP(c, hipStreamSynchronize(c->stream));
  read_counters(c, hm, ht);
  *maxd = std::sqrt(c->nb_host->d2);
  for (int k = 0; k < 5; ++k) {
    c->ell[k].width = hm[k];
    if (k < 4) {
      c->ell[k].owidth = hm[5 + k];
      c->ell[k].rwidth = hm[9 + k];
    }
  }
  return A2C_OK;
}

double skin_length() {
  static const double skin = [] {
    const char* e = std::getenv("A2C_NBR_SKIN");
    const double v = e ? std::atof(e) : 0.2;
    return v > 0.0 ? v : 0.0;
  }();
  return skin;
}

}  // namespace

// Host driver.  The positions are the context state c->dX (on the device).
// First build: the cell walk at rc.  Later builds: lists at rc + skin by
// the cell walk, kept with the positions they were built at, and the lists
// at rc filtered from them -- again at the next builds while no site has
// moved by skin/2 (a pair within rc now was within rc + skin then).
int nbr_build(a2c_fe_ctx* c) {
  const int N = c->N;
  const double rc = c->desc.rc, skin = skin_length();
  int hm[16] = {0};
  unsigned long long ht[5] = {0, 0, 0, 0, 0};
  bool refreshed = false;
  double maxd = 0.0;
  if (int rc2 = nbr_counters(c)) return rc2;
  if (c->nb_sup_ok) {
    if (int rc2 = refresh(c, true, hm, ht, &maxd)) return rc2;
    refreshed = 2.0 * maxd < skin * (1.0 - 1e-9);  // else the filtered lists may miss a pair
    c->nb_sup_ok = refreshed;
  }
  bool fits = skin > 0.0 && !c->nb_sup_off && c->nb_builds > 0;
  for (int ax = 0; ax < 3; ++ax)
    if (c->desc.periodic[ax] && c->desc.box[ax] < 2.0 * (rc + skin)) fits = false;
  if (!refreshed && fits) {  // new skin lists, then the lists at rc filtered from them
    unsigned long long hs[5];
    const int rc2 = walk_cells(c, rc + skin, c->nb_sup, false, hm, hs);
    if (rc2 == A2C_OK) {
      if (int rc3 = size_skin_extras(c)) return rc3;
      if (!c->nb_sup_q) A2C_HIP(c, dmalloc(&c->nb_sup_q, 32 * (size_t)std::max(N, 1)));
      A2C_HIP(c, hipMemcpyAsync(c->nb_sup_q, c->dX, 32 * (size_t)N, hipMemcpyDeviceToDevice, c->stream));
      if (int rc3 = refresh(c, false, hm, ht, &maxd)) return rc3;
      c->nb_sup_ok = refreshed = true;
      maxd = 0.0;
    } else if (rc2 == A2C_ENBR_OVERFLOW) {
      c->nb_sup_off = true;  // rows over the cap at rc + skin: walk the cells at rc from now on
    } else {
      return rc2;
    }
  }
  if (!refreshed) {
    const int rc2 = walk_cells(c, rc, c->ell, true, hm, ht);
    if (rc2 == A2C_ENBR_OVERFLOW) {
      c->have_nbr = false;
      return set_err(c, A2C_ENBR_OVERFLOW, "a site has more neighbors than max_neighbors");
    }
    if (rc2) return rc2;
    ++c->nb_builds;
  }
  if (!c->depair) A2C_HIP(c, dmalloc(&c->depair, sizeof(double) * std::max(N, 1)));
  c->stats.max_neib = hm[13];
  for (int w = 0; w < 5; ++w) {
    c->stats.width[w] = hm[w];
    c->stats.total[w] = (int64_t)ht[w];
  }
  c->stats.refreshed = refreshed ? 1 : 0;
  c->stats.max_displacement = maxd;
  c->have_nbr = true;
  c->lat_dirty = true;
  return A2C_OK;
}

void free_pair_buffers(Ell& L) {
  (void)dfree(L.ocnt); (void)dfree(L.rcnt); (void)dfree(L.oj); (void)dfree(L.orv);
  (void)dfree(L.rbuf);
  L.ocnt = L.rcnt = L.oj = L.orv = nullptr;
  L.rbuf = nullptr;
  L.ocap = L.bcap = 0;
  L.owidth = L.rwidth = 0;
}

}  // namespace a2c
