// Internal declarations shared by the HIP sources of liba2c_fe.so.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "a2c_fe.h"

namespace a2c {

// Device buffers of the library (devmem.cpp): a caching allocator with
// hipMalloc/hipFree semantics (dfree synchronises the block's device first).
hipError_t dmalloc(void** ptr, size_t bytes);
template <class T>
inline hipError_t dmalloc(T** ptr, size_t bytes) {
  return dmalloc(reinterpret_cast<void**>(ptr), bytes);
}
hipError_t dfree(const void* ptr);
hipError_t hmalloc(void** ptr, size_t bytes);  // pinned host staging, cached alike
template <class T>
inline hipError_t hmalloc(T** ptr, size_t bytes) {
  return hmalloc(reinterpret_cast<void**>(ptr), bytes);
}
hipError_t hfree(const void* ptr);
// While one lives, this thread's current device is the given one: what a context
// makes at its first use (memory, events) belongs to the context's device,
// whichever is current in the calling thread.
class DeviceScope {
 public:
  explicit DeviceScope(int device);
  ~DeviceScope();
  DeviceScope(const DeviceScope&) = delete;
  DeviceScope& operator=(const DeviceScope&) = delete;
  hipError_t status() const { return err_; }

 private:
  int prev_ = -1;  // the device to go back to, -1 if it is the given one
  hipError_t err_;
};
// While one lives, this thread's releases on its device (dfree, hfree) do not
// wait for the device again: it waited when it was made, and nothing that uses
// the released blocks is issued during its life (a context's teardown, ~50
// blocks at ~1 us each).
class ReleaseScope {
 public:
  explicit ReleaseScope(int device);
  ~ReleaseScope();
  ReleaseScope(const ReleaseScope&) = delete;
  ReleaseScope& operator=(const ReleaseScope&) = delete;

 private:
  int prev_;
};

// Transfers between pageable memory of a caller and the device through pinned
// staging, in parts, so that the copy on the host and the transfer overlap.  stage
// (cap bytes, a multiple of 16) must be idle.  Device buffers are the library's own
// (whole 16-byte words).  upload returns with transfers in flight from stage
// unless it had to reuse it; download returns when dst is complete.  A kernel writes
// the pinned words: for the small transfers that is ~20 us sooner than the
// copy engine, for large ones as fast.
class HostTransfer {
 public:
  hipError_t upload(hipStream_t st, char* stage, size_t cap, void* ddst, const void* src, size_t bytes);
  hipError_t download(hipStream_t st, char* stage, size_t cap, void* dst, const void* dsrc, size_t bytes);
  ~HostTransfer();

 private:
  static constexpr int PARTS = 8;
  static constexpr size_t PART_MIN = (size_t)512 << 10;
  hipEvent_t ev_[PARTS] = {};
};
// device words to pinned memory by a kernel on st, rounded up to 16 bytes
hipError_t copy_to_pinned(hipStream_t st, void* pinned, const void* dsrc, size_t bytes);

constexpr double KB = 8.6173324e-5;  // Boltzmann constant, eV/K (minimizer.cpp:92)
constexpr int NBR_CAP = 256;          // per-site neighbor cap of the build kernel

// Row order of the pair-once evaluation.  An FCC crystal lists its sites cell
// by cell, four to a cell, and the four see their neighbors in different
// directions: 64 consecutive sites at the same list slot gather from 64
// scattered places.  The split lists, the shares and the per-site arrays the
// pair passes read are therefore kept with every fourth site together -- the
// first site of all cells, then the second, ... (rows past the last whole
// group of four keep their place) -- so a wave's 64 rows are the same site of
// 64 consecutive cells: slot t of all of them is the same neighbor vector, the
// neighbors are consecutive rows too, and gathers and share stores touch 8 to
// 16 cache lines instead of 64, and shares fill whole lines.  (40^3 cells, mixed:
// k_dens_own 211 -> 170 us, k_grad_own 355 -> 280 us; k_rows costs 14 us.)  Any
// other site order only loses that: this is a permutation of each species' rows.
__host__ __device__ inline int row_of_site(int r, int rows) {
  const int q = rows >> 2;
  return r < 4 * q ? (r & 3) * q + (r >> 2) : r;
}
__host__ __device__ inline int site_of_row(int p, int rows) {
  const int q = rows >> 2;
  if (p >= 4 * q) return p;
  const int b = (p >= q) + (p >= 2 * q) + (p >= 3 * q);
  return (p - b * q) * 4 + b;
}

// One neighbor list in ELL layout: entry t of row r is idx[t * rows + r], so
// lane r of a wave reading slot t touches consecutive words (coalesced).
// Indices are species-local (Pd index or H index), rows sorted ascending.
struct Ell {
  int32_t rows = 0;
  int32_t width = 0;
  int32_t* idx = nullptr;  // width * rows
  int32_t* cnt = nullptr;  // rows
  // Pair-once evaluation (each unordered pair evaluated once, by its owner).
  // Rows and neighbor indices of this part are in row order (row_of_site).
  // Every row is split, keeping its order, into the entries this row owns
  // and the entries it receives; both halves are compact (slot-major, no
  // gaps), so a wave's lanes step through their halves without masking each
  // other off.  Widths are the longest half over all rows.
  int32_t owidth = 0, rwidth = 0;
  int32_t* ocnt = nullptr;  // rows: owned entries
  int32_t* oj = nullptr;    // owidth * rows: neighbor of owned entry t
  int32_t* orv = nullptr;   // owidth * rows: slot of the pair in the partner's received half
  int32_t* rcnt = nullptr;  // rows: received entries
  // Received shares, written by the partner's owner pass (already weighted
  // by the partner's occupancy) and summed by this row's receive pass of the
  // same evaluation: rwidth * rows entries of a float (density) or float4
  // (gradient) in the mixed passes, a double or double4 in the FP64 passes --
  // one buffer serves all four.  During the build it holds the received
  // half's site indices.
  void* rbuf = nullptr;
  int64_t ocap = 0;            // allocated entries of oj/orv
  int64_t bcap = 0;            // allocated bytes of rbuf
  int64_t cap = 0;             // allocated entries of idx (grow-only across rebuilds)
};

// Device view of one lattice: what every kernel needs.  The eval kernels
// read it from device memory through a block -> lattice map, so one launch
// covers any set of lattices (a batch) and a single lattice is a batch of one.
// Each lattice's sites are split into blocks of 256 starting at its site 0 in
// every launch, so its results do not depend on the other lattices present.
struct LatDev {
  int32_t npd = 0, nh = 0;
  int32_t periodic[3] = {0, 0, 0};
  int32_t blk0 = 0;          // first block of this lattice in the current launch
  int32_t kl32 = 1, kl64 = 1;    // lanes per site in the mixed / FP64 pair-owner passes
  int32_t owg0_32 = 0, owg0_64 = 0;  // first workgroup of this lattice in those launches
  double box[3] = {0, 0, 0};
  double ibox[3] = {0, 0, 0};  // 1/box: the image shift of a listed pair is L*rint(d/L) with d/L as d*(1/L)
  double T = 0;
  int32_t rule = 0;          // A2C_QUAD_R12 or A2C_QUAD_GH3
  Ell pdpd, pdh, hpd, hh, hh1;
  const double* X = nullptr;  // 4N state (32-byte aligned)
  double* G = nullptr;        // 4N gradient
  const double* x = nullptr;  // nh occupancy
  double* rho = nullptr;      // N densities
  double* Fp = nullptr;       // N F'(rho) (FP64 path)
  float2* aux = nullptr;      // N {F'(rho), x} (mixed path)
  double* emb = nullptr;      // N embedding energy (x-weighted for H)
  double* epair = nullptr;    // N pair-energy partial (mixed path)
  const double* w = nullptr;  // 4N direction (site order), or null: the gradient receive pass then also sums
  double* slope = nullptr;    // G . w into slope
  double* part = nullptr;     // block partial sums of f and G . w: one of each per 256 sites, or per 64 (recv_lanes)
  int32_t* done = nullptr;    // blocks of the gradient receive pass that have put theirs (k_rows clears it)
  int32_t rl = 1;             // lanes per row in the receive passes (recv_lanes)
  double* f = nullptr;        // objective
  // pair-once evaluation, per species in row order (Pd rows, then H rows; rho,
  // Fp, aux, emb and epair are in this order too while it runs):
  double2* qxy = nullptr;     // N {x, y} and
  double2* qzs = nullptr;     // N {z, sigma}: two 16-byte arrays, each gathered whole lines at a time
  double* xrow = nullptr;     // nh occupancy
  double4* gown = nullptr;    // N gradient sums of the owned pairs
};
using DevSys = LatDev;
constexpr int SITE_BLOCK = 256;  // sites per block of every site-parallel kernel
__host__ __device__ inline int site_blocks(int n) { return (n + SITE_BLOCK - 1) / SITE_BLOCK; }
// Blocks of a lattice in a launch that must write its results even if it has no
// sites (zeros then).
__host__ __device__ inline int lattice_blocks(int n) { return n > 0 ? site_blocks(n) : 1; }

// Lanes per row of the receive passes.  Up to RECV_SPLIT_SITES a pass is bound by
// the memory latency of one row's ~20 shares per list, and RECV_LANES lanes
// take them in turn; beyond, it streams, and one lane per row reads whole
// lines.  Mixed gradient pass, 1 / 4 lanes: 1,728 sites 16.5 / 9.9 us, 21,952
// sites 17.0 / 13.7, 46,656 sites 17.8 / 20.3, 512,000 sites 90 / 131; FP64 16.0 /
// 11.3, 17.3 / 15.3, 18.4 / 23.1, 174 / 186.
constexpr int RECV_LANES = 4, RECV_SPLIT_SITES = 32768;
__host__ __device__ inline int recv_lanes(int n) { return n <= RECV_SPLIT_SITES ? RECV_LANES : 1; }

// Global-memory views.  Pointers read from a descriptor in memory are
// generic to the compiler, which then issues flat_* instructions: those count
// against the LDS counter as well as the vector-memory one, so every wait for
// a table lookup also waits out outstanding gathers and stores.  Loads and
// stores through these views are global_* instructions.
#if defined(__HIP_DEVICE_COMPILE__)
#define A2C_GLOBAL __attribute__((address_space(1)))
#else
#define A2C_GLOBAL  // the host pass of a .hip file compiles device code too, without address spaces
#endif
template <class T>
__device__ __forceinline__ A2C_GLOBAL T* gmem(T* p) {
  return (A2C_GLOBAL T*)p;
}

// The shares ph, ph + G, ... of the n received by one row of a slot-major
// buffer (share t at base[t * rows + row]) passed to add in slot order.  The
// loads of RU of them are issued before any is added, so a row costs one
// memory latency per RU shares rather than one per share; the order of the
// additions, and so the result, is that of a plain loop.
template <int RU, class T, class Add>
__device__ __forceinline__ void for_row_shares(const A2C_GLOBAL T* __restrict__ base, size_t rows, int row, int n,
                                               int ph, int G, Add add) {
  for (int t = ph; t < n; t += RU * G) {
    T v[RU];
#pragma unroll
    for (int u = 0; u < RU; ++u)
      if (t + u * G < n) v[u] = base[(size_t)(t + u * G) * rows + row];
#pragma unroll
    for (int u = 0; u < RU; ++u)
      if (t + u * G < n) add(v[u]);
  }
}
// Loads in flight per lane with one lane per row: 8 for the density pass's
// scalar shares (faster at every size measured), 2 for the gradient pass's
// shares of 16 or 32 bytes (a 40^3-cell lattice, streaming at HBM speed: RU =
// 1/2/4/8 took 74.6/76.3/83.0/87.9 us, where the registers they hold cost
// waves).  With RECV_LANES lanes per row 6, a lane's part of ~20, or 3 of 32 bytes.
constexpr int RECV_RU_SCALAR = 8, RECV_RU_WIDE = 2, RECV_RU_SPLIT = 6;
template <int RU, class T, class Add>
__device__ __forceinline__ void row_shares(const Ell& L, int row, int ph, int G, Add add) {
  const A2C_GLOBAL T* base = gmem(reinterpret_cast<const T*>(L.rbuf));
  const int n = L.rcnt[row];
  if (G == 1) for_row_shares<RU>(base, L.rows, row, n, 0, 1, add);
  else for_row_shares<(sizeof(T) > 16 ? RECV_RU_SPLIT / 2 : RECV_RU_SPLIT)>(base, L.rows, row, n, ph, G, add);
}

// Place of a lane in a receive pass: rq blocks of 256 lanes per 256 rows, of
// which a lattice with one lane per row uses the first.
struct RecvLane {
  int lb, q, G;  // block of 256 rows within the lattice, quarter of it, lanes per row
  int s, ph;     // row (row order) and phase
  bool idle;     // a block without work
  __device__ __forceinline__ RecvLane(const LatDev& S, int lblk, int quarter)
      : lb(lblk), q(quarter), G(S.rl), ph(0), idle(false) {
    const int t = threadIdx.x;
    if (G == 1) {
      idle = q != 0;
      s = lb * SITE_BLOCK + t;
    } else {
      s = lb * SITE_BLOCK + q * (SITE_BLOCK / RECV_LANES) + t / RECV_LANES;
      ph = t % RECV_LANES;
    }
  }
  __device__ __forceinline__ double sum(double v) const { return G == 1 ? v : site_sum_row(v); }
  static __device__ __forceinline__ double site_sum_row(double v) {
#pragma unroll
    for (int off = RECV_LANES / 2; off > 0; off >>= 1) v += __shfl_down(v, off, RECV_LANES);
    return v;
  }
};

// Lanes per site of the pair-owner passes.  A small lattice gives too few
// waves to fill the GPU with one lane per site, and each lane would walk its
// ~40 owned pairs x 12 points serially; splitting a site's pairs over K lanes
// (combined in a fixed shuffle order) cuts that latency K-fold.  Large
// lattices already fill the GPU in a batch, where one lane per site keeps the
// neighbor-list loads coalesced.  K comes from the process-wide table of
// a2c_tune.h (lattice size class and precision), so it depends only on the
// lattice: its results are the same in any batch.
int lanes_per_site(int n_sites, bool fp64);
constexpr int MAX_LANES_PER_SITE = 16;
// Workgroup units of a pair-owner pass: 256 lanes each, the rows of one species
// per unit (Pd units first), so that everything that depends on the species --
// list pointers, pair kind, weights -- is uniform and stays in scalar
// registers.
__host__ __device__ inline int owner_units(int rows, int K) {
  return (int)(((int64_t)rows * K + SITE_BLOCK - 1) / SITE_BLOCK);
}
__host__ __device__ inline int owner_units(int npd, int nh, int K) { return owner_units(npd, K) + owner_units(nh, K); }

// Fixed-order sum over the K lanes of a site (K a power of two <= 64, lanes
// contiguous within a wave); the total lands in the group's first lane.
template <typename T>
__device__ inline T site_sum(T v, int K) {
  for (int off = K >> 1; off > 0; off >>= 1) v += __shfl_down(v, off, K);
  return v;
}

// 3-point Gauss-Hermite product rule on the relative coordinate: per axis
// nodes -sqrt(3), 0, sqrt(3) (standard normal), weights 1/6, 2/3, 1/6.
// Node k in 0..26 has per-axis offsets a_c = (k / 3^c) % 3 - 1, so
// z = sqrt(3) a and weight w = prod_c gh_w(a_c).  The nodes of one pair are
// r_k = d + s z_k with s = sqrt(sigma_i^2 + sigma_j^2), and
// dr_k/dsigma_i = z_k sigma_i / s.
constexpr double GH_Z = 1.7320508075688772935;
__host__ __device__ constexpr double gh_w(int a) { return a == 0 ? 2.0 / 3.0 : 1.0 / 6.0; }
__device__ inline void gh_node(int k, double z[3], double& w) {
  const int a0 = k % 3 - 1, a1 = (k / 3) % 3 - 1, a2 = k / 9 - 1;
  z[0] = GH_Z * a0;
  z[1] = GH_Z * a1;
  z[2] = GH_Z * a2;
  w = gh_w(a0) * gh_w(a1) * gh_w(a2);
}


// General model of a context (a2c_fe_set_potential_*, a2c_fe_set_quadrature):
// the functions of a tabulated potential as cubic pieces on uniform grids,
// and the rule as a node table.  Function order: F_Pd, F_H (embedding),
// f_Pd, f_H (density), r phi_PdPd, r phi_PdH, r phi_HH (pair).
enum { GEN_F_PD = 0, GEN_F_H, GEN_RHO_PD, GEN_RHO_H, GEN_RPHI_PD, GEN_RPHI_PDH, GEN_RPHI_H, GEN_NFN };
// An embedding function: cubic pieces on its grid.
struct GenFn {
  int32_t n = 0;        // nodes (n - 1 pieces), node k at k * h
  int32_t off = 0;      // first piece in the coefficient array
  double ih = 0.0;      // 1 / h
  double yend = 0.0;    // value and slope at the last node (the function
  double dend = 0.0;    // continues along it)
};
// The five r-functions share one grid and one table row per node (80 bytes),
// so that a radius is located once and the two or three functions a pair needs
// lie next to each other: r phi_PdPd f_Pd | r phi_PdH | f_H r phi_HH.
enum { GEN_S_RPHI_PD = 0, GEN_S_RHO_PD, GEN_S_RPHI_PDH, GEN_S_RHO_H, GEN_S_RPHI_H, GEN_NS };
template <class E>
struct GenR {
  const E* row = nullptr;  // GEN_NS entries per node (pieces: per interval, plus one unused row)
  int32_t n = 0;           // nodes
  double ih = 0.0;         // 1 / h
};
struct GenDev {
  int32_t pot = 0;      // 0: compiled-in Pd-H closed forms; 1: tabulated
  int32_t K = 0;        // nodes of the rule
  int32_t rel = 0;      // 1: nodes z on the relative coordinate, r = d + s z,
                        //    s^2 = sigma_i^2 + sigma_j^2 (the Gauss-Hermite rule);
                        // 0: 6-D nodes, r = d + sqrt(2) (sigma_i xi1 - sigma_j xi2)
  const double* nodes = nullptr;  // K x 8: xi1[3] (or z), xi2[3], w, 0
  const double4* tab = nullptr;   // embedding pieces (c0..c3 in u = x/h - k)
  GenFn fn[2];                    // GEN_F_PD, GEN_F_H
  GenR<double2> r64;  // FP64: node value and slope (times h); the pieces' coefficients follow from two nodes
  GenR<float4> r32;   // FP32 (mixed): c0..c3 of each piece, rounded from FP64
};

// Minimum-image geometry of one lattice, copied out of its descriptor into
// registers before a pair loop (the loop's stores could otherwise alias the
// descriptor, and its fields would be reloaded for every pair).
struct Image {
  double box[3], ibox[3];
  double half[3];  // L / 2 on a periodic axis, else infinity
};
__device__ __forceinline__ Image image_of(const LatDev& S) {
  Image g;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    g.box[c] = S.box[c];
    g.ibox[c] = S.ibox[c];
    g.half[c] = S.periodic[c] ? 0.5 * S.box[c] : __builtin_huge_val();
  }
  return g;
}
// d = q_i - image(q_j): a periodic axis shifts q_j by L rint((q_j - q_i) / L).
// A listed pair is within rc <= L/2 of an image, so the shift is zero unless
// |q_i - q_j| > L/2 -- no pair of most waves, which then skip it.
__device__ __forceinline__ void image_vec(const Image& g, const double qi[3], const double qj[3], double d[3]) {
  bool far = false;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    d[c] = qi[c] - qj[c];
    far |= fabs(d[c]) > g.half[c];
  }
  if (far) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (fabs(d[c]) > g.half[c]) d[c] = qi[c] - fma(-g.box[c], rint((qj[c] - qi[c]) * g.ibox[c]), qj[c]);
  }
}

// Place of a lane in a pair-owner pass: its row (row order) and its phase ph
// among the row's K lanes, which take owned slots ph, ph + K, ...  u: the
// wave's unit within the lattice (uniform).
struct OwnerLane {
  bool pd;   // uniform
  int rows;  // of the species
  int row, ph;
  __device__ __forceinline__ OwnerLane(const LatDev& S, int u, int K) {
    const int up = owner_units(S.npd, K), sh = 31 - __builtin_clz(K);
    pd = u < up;
    rows = pd ? S.npd : S.nh;
    const int lane = (int)threadIdx.x % SITE_BLOCK;
    ph = lane & (K - 1);
    row = (pd ? u : u - up) * (SITE_BLOCK >> sh) + (lane >> sh);
  }
};

// Logical site block of a workgroup.  Workgroups are dealt to the 8 XCDs
// round-robin by index; this bijection gives XCD k one contiguous range of
// site blocks, so the neighbor data its waves gather stays within its own L2
// instead of every XCD touching the whole lattice.
constexpr int NUM_XCD = 8;
__device__ inline int xcd_block() {
  const int b = blockIdx.x, n = gridDim.x;
  const int x = b % NUM_XCD, q = n / NUM_XCD, r = n % NUM_XCD;
  return x * q + (x < r ? x : r) + b / NUM_XCD;
}

// Block partials summed by the block of their group that arrives last, instead of
// by a launch of its own (~4 us and a gap for a few kilobytes).  Thread 0 puts its
// block's partials with put_part, then the whole block calls last_block; where
// it returns true, every partial of the group's n blocks is visible to get_part
// (device-scope accesses, which pass the XCDs' separate L2s by; the wait orders the
// partials before the count without writing those caches back).  sum_parts adds
// in an order that depends on n alone.  done starts at 0.
__device__ __forceinline__ void put_part(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get_part(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool last_block(int32_t* done, int n) {
  __shared__ int last;
  if (threadIdx.x == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
  }
  __syncthreads();
  return last != 0;
}
// out(k, sum of part[k stride + j], j < n) for k < K, by a block of SITE_BLOCK:
// wave w takes k = w, w + 4, ..., all of its sums' loads and trees in flight
// together.
template <int K, class Out>
__device__ __forceinline__ void sum_parts(const double* part, size_t stride, int n, Out out) {
  constexpr int W = SITE_BLOCK / 64, KW = (K + W - 1) / W, U = KW > 4 ? 1 : 8 / KW;  // sums per wave, loads per sum
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double v[KW] = {};
  for (int j0 = lane; j0 < n; j0 += 64 * U) {
    double p[KW][U];
#pragma unroll
    for (int i = 0; i < KW; ++i)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = w + W * i, j = j0 + 64 * u;
        p[i][u] = k < K && j < n ? get_part(part + k * stride + j) : 0.0;
      }
#pragma unroll
    for (int i = 0; i < KW; ++i)
#pragma unroll
      for (int u = 0; u < U; ++u) v[i] += p[i][u];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < KW; ++i) v[i] += __shfl_down(v[i], off);
#pragma unroll
  for (int i = 0; i < KW; ++i)
    if (lane == 0 && w + W * i < K) out(w + W * i, v[i]);
}

// End of a gradient receive pass: the block's sums of fs and sl, and of all blocks'
// sums by the last one, into the objective and (S.w) the slope.  Every lane of a
// working block calls it.
__device__ __forceinline__ void finish_objective(const LatDev& S, const RecvLane& ln, double fs, double sl) {
  __shared__ double red[2][SITE_BLOCK / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    fs += __shfl_down(fs, off);
    sl += __shfl_down(sl, off);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = fs;
    red[1][threadIdx.x >> 6] = sl;
  }
  __syncthreads();
  const int n = (ln.G == 1 ? 1 : RECV_LANES) * lattice_blocks(S.npd + S.nh);
  if (threadIdx.x == 0) {
    double* p = S.part + (ln.G == 1 ? ln.lb : RECV_LANES * ln.lb + ln.q);
    put_part(p, (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]));
    if (S.w) put_part(p + n, (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
  }
  if (!last_block(S.done, n)) return;
  if (S.w) sum_parts<2>(S.part, n, n, [&](int k, double v) { *(k ? S.slope : S.f) = v; });
  else sum_parts<1>(S.part, 0, n, [&](int, double v) { *S.f = v; });
}
// G . w of one site
__device__ __forceinline__ double site_slope(const LatDev& S, size_t site, double g0, double g1, double g2, double g3) {
  if (!S.w) return 0.0;
  const A2C_GLOBAL double* w = gmem(S.w) + 4 * site;
  return (g0 * w[0] + g1 * w[1]) + (g2 * w[2] + g3 * w[3]);
}

// What a neighbor build tells the host: the 14 maxima and the overflow flag of
// the count pass (nbr.hip), list totals, squared largest displacement.
struct NbrCounters {
  int32_t max[16];
  unsigned long long total[5];
  double d2;
};

struct Timing;

// a2c_fe_create on a stream of the caller's (a batch's own lattices share
// its stream: creating and destroying one per lattice cost ~1.3 ms), or on a
// stream of its own when shared is null
int fe_create(const a2c_fe_desc* desc, hipStream_t shared, a2c_fe_ctx** out);

}  // namespace a2c

struct a2c_fe_ctx {
  a2c_fe_desc desc;
  int32_t N = 0;
  bool own_stream = true;
  hipStream_t stream = nullptr;
  std::string err;

  // state
  double* dX = nullptr;      // 4N
  double* dG = nullptr;      // 4N
  double* dx = nullptr;      // nH occupancy
  double* drho = nullptr;    // N
  double* dFp = nullptr;     // N  F'(rho)
  double* demb = nullptr;    // N  embedding energy per site (x-weighted for H)
  double* depair = nullptr;  // N  pair-energy partial of the mixed path
  double* dpart = nullptr;   // block partial sums
  double* dF = nullptr;      // 1 objective, in pinned memory that the kernels write
  int32_t nblk_red = 0;
  bool have_x = false;
  bool have_nbr = false;

  // neighbor lists
  a2c::Ell ell[5];           // PdPd, PdH, HPd, HH, HH1
  // neighbor-build scratch (grow-only)
  int* nb_cid = nullptr;     // N: cell of each site
  void* nb_order = nullptr;  // N double4: positions in cell order, site index in .w
  int* nb_cc = nullptr;      // cells + 1: cell starts
  int* nb_cursor = nullptr;  // cells + 1: histogram, then placement cursors
  a2c::NbrCounters* nb_host = nullptr;  // pinned: the reduced counters
  int* nb_misc = nullptr;    // build counters (list widths, totals; copies per workgroup group), displacement, bounding box
  int64_t nb_cap_cells = 0;
  // skin lists: the pair lists at rc + skin and the positions they were built
  // at; while every site is within skin/2 of those positions the lists at rc
  // are filtered from them (nbr.hip)
  a2c::Ell nb_sup[5];
  double* nb_sup_q = nullptr;  // 4N: positions at the skin build
  bool nb_sup_ok = false;      // skin lists valid for the current positions' neighbors
  bool nb_sup_off = false;     // skin lists refused for this context (a row over the cap)
  int32_t nb_builds = 0;       // builds by walking the cells
  int32_t* dpdpdnum = nullptr;  // nPd*3
  a2c_nbr_stats stats{};

  // mixed-precision tables + FP32 mirrors
  float4* dtab = nullptr;    // cubic coefficient tables (5 x 500 intervals)
  double* dtab64 = nullptr;  // FP64 polynomial tables of the exponential functions
  float2* daux = nullptr;    // per site {F'(rho), x} in FP32
  double2* dqxy = nullptr;   // row-order copies of the state and occupancy, and the
  double2* dqzs = nullptr;   // owned pairs' gradient sums (pair-once evaluation)
  double* dxrow = nullptr;
  double4* dgown = nullptr;

  // launch descriptors: this context is a batch of one lattice
  a2c::LatDev* hlat = nullptr;   // pinned host copy
  a2c::LatDev* dlat = nullptr;   // device copy
  int32_t* db2l = nullptr;       // block -> lattice (all zero)
  bool lat_dirty = true;

  // host staging (pinned)
  double* hX = nullptr;
  double* hG = nullptr;
  a2c::HostTransfer xfer;

  // occupancy scratch of the chemical potential and the diffusion step
  // (allocated at their first call, kept for the context's lifetime)
  double* occ_g = nullptr;     // nH gamma
  int32_t* occ_full = nullptr; // nH full_H
  double* occ_corr = nullptr;  // N correction sums
  double* occ_uv = nullptr;    // 2 nH edge-term factors of the diffusion step
  double* occ_xn = nullptr;    // nH new occupancy
  double* occ_part = nullptr;  // 4 per block of the balance
  double* occ_bal = nullptr;   // 4: the balance of the last step (a2c_diffusion_balance)
  a2c_diffusion_balance last_balance{};

  // general model (null gen_nodes: the descriptor's rule and the closed forms)
  bool gen_on = false;          // evaluate with the general kernels
  bool gen_table_rule = false;  // a node table was set (else the descriptor's rule)
  a2c::GenDev gen{};
  double* gen_nodes = nullptr;  // device: K x 8
  double4* gen_tab = nullptr;   // device: embedding pieces
  double2* gen_r64 = nullptr;   // device: r-functions, FP64
  float4* gen_r32 = nullptr;    // device: r-functions, FP32
  size_t gen_tab_n = 0, gen_r64_n = 0, gen_r32_n = 0;

  a2c::DevSys sys() const {
    a2c::DevSys s;
    s.npd = desc.n_pd;
    s.nh = desc.n_h;
    for (int c = 0; c < 3; ++c) {
      s.box[c] = desc.box[c];
      s.ibox[c] = desc.box[c] > 0.0 ? 1.0 / desc.box[c] : 0.0;
      s.periodic[c] = desc.periodic[c];
    }
    s.T = desc.temperature;
    s.rule = desc.quad_rule;
    s.pdpd = ell[0]; s.pdh = ell[1]; s.hpd = ell[2]; s.hh = ell[3]; s.hh1 = ell[4];
    s.x = dx; s.rho = drho; s.Fp = dFp; s.aux = daux; s.emb = demb; s.part = dpart; s.epair = depair;
    s.done = reinterpret_cast<int32_t*>(dpart + 2 * (size_t)a2c::RECV_LANES * nblk_red);
    s.rl = a2c::recv_lanes(N);
    s.qxy = dqxy; s.qzs = dqzs; s.xrow = dxrow; s.gown = dgown;
    return s;
  }
};

namespace a2c {

// error helpers -------------------------------------------------------------
int set_err(a2c_fe_ctx* c, int code, const std::string& msg);
#define A2C_HIP(ctx, call)                                                       \
  do {                                                                           \
    hipError_t e_ = (call);                                                      \
    if (e_ != hipSuccess)                                                        \
      return ::a2c::set_err((ctx), A2C_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

// kernels (launchers) ---------------------------------------------------------
int nbr_build(a2c_fe_ctx* c);                           // nbr.hip
void free_pair_buffers(Ell& L);                         // nbr.hip
// Multi-lattice launches: lats/b2l on the device, nblk = total site blocks,
// nlat = lattices.  The FP64 path fills rho, Fp, emb, G, part, f; the mixed
// path rho, aux, emb, G, part, f.
struct Launch {
  const LatDev* lats;
  const int32_t* b2l;
  int nblk, nlat;
  int rq = 1;  // blocks per site block in the receive passes: RECV_LANES if some lattice takes that many
  hipStream_t stream;
  int deriv_mode;
  double fd_eps;
  const float4* tab;  // mixed path
  const double* tab64 = nullptr;  // FP64 pair-owner passes
  const int32_t* ob2l = nullptr;  // pair-owner workgroup -> lattice
  int onblk = 0;                  // pair-owner workgroups
  bool mixed_full = false;    // mixed path: every pair from both ends (A/B reference)
  bool full_pairs64 = false;  // FP64 analytic path: every pair from both ends (A/B reference)
  bool empty = false;         // some lattice of the launch has no sites
  int rules = 1;              // bit r set: some lattice of the launch uses quadrature rule r
};
bool mixed_full_pairs();  // A2C_MIXED_PAIRS=full selects the both-ends kernels
bool fp64_full_pairs();   // A2C_FP64_PAIRS=full likewise for the FP64 kernels
int run_eval64(const Launch& L, Timing* tm);
int run_eval32(const Launch& L, Timing* tm);
int run_final_sum(const Launch& L);
bool fold_rows(const Launch& L);  // the density pass makes the row-order copies itself (pair_rows.hpp)
int run_rows(const Launch& L);  // row-order copies of state and occupancy (pair-once evaluation)
int sync_lattice(a2c_fe_ctx* c, const double* dX, double* dG, double* dF);  // refresh the one-lattice descriptor
int launch_eval64(a2c_fe_ctx* c, const double* dX, double* dG, double* dF, bool timed, Timing* tm);
int launch_density64(a2c_fe_ctx* c, const double* dX, bool by_site);  // fills drho, dFp, demb
// Chemical potential of the H sites: gamma and full in site order, corr
// (k_chem_pre) in row order.
struct ChemArgs {
  const double* corr;
  double ch[4];
  double gamma_bd;
  double* gamma;
  int32_t* full;
};
int launch_chem64(a2c_fe_ctx* c, const ChemArgs& a);  // after launch_density64 in row order
int launch_eval32(a2c_fe_ctx* c, const double* dX, double* dG, double* dF, bool timed, Timing* tm);
int build_tables(a2c_fe_ctx* c);                        // eval32.hip
int tables_download(a2c_fe_ctx* c, float* out);         // 5*500 float4
void host_tables(std::vector<float4>& t);              // FP32 cubic tables in r (host)
void host_tables_s(std::vector<float4>& t);            // appends the FP32 cubic tables in |r|^2
// FP64 tables of the EAM functions in r (exported; no kernel reads them): per function T64_N intervals of 0.05 A
// over [1, 6) A, each a polynomial in the local coordinate u in [0, 1).  Part
// one: the exponential functions (f_H, phi_PdH, phi_H), degree T64_D, T64_P
// doubles per row (c0..c8, one pad); part two, after it: the Pd polynomials
// (f_Pd, phi_Pd), degree T64Q_D, T64Q_P doubles per row (c0..c11).
constexpr int T64_N = 100, T64_D = 8, T64_P = 10, T64_NF = 3;
enum { T64_FH = 0, T64_PHPDH = 1, T64_PHH = 2 };
constexpr int T64Q_D = 11, T64Q_P = 12, T64Q_NF = 2;
enum { T64Q_FPD = 0, T64Q_PHPD = 1 };
constexpr int T64_PART1 = T64_NF * T64_N * T64_P;                // doubles
constexpr int T64_SIZE = T64_PART1 + T64Q_NF * T64_N * T64Q_P;  // doubles
void host_tables64(std::vector<double>& t);
void pass_eval64(const std::vector<double>& t, int fn, double r, double& v, double& d);
double pass_eval32(const std::vector<float4>& t, int fn, double r, double& v, double& d);  // returns the radius
void host_tables64_s(std::vector<double>& t);  // those of the FP64 owner passes, in |r|^2 (eval64.hip)
// The FP32 and FP64 EAM tables on one device, uploaded at the first call for
// that device and shared by every context and batch of the process until it
// ends (they depend on nothing but the compiled-in potential); never freed.
struct DeviceTables {
  float4* t32 = nullptr;
  double* t64 = nullptr;
};
hipError_t device_tables(int device, DeviceTables* out);
int host_staging(a2c_fe_ctx* c);  // pinned hX, hG of the host-array entry points (capi.cpp)
int upload_state(a2c_fe_ctx* c, const double* X);  // X to the context state dX through hX, on the context stream
int download_state(a2c_fe_ctx* c, double* out, const double* dsrc);  // 4N doubles through hG; complete on return
// General model (evalgen.hip, general.cpp)
int run_eval_gen(const LatDev* dlat, int npd, int nh, const GenDev& g, int deriv_mode, double eps, bool fp32, hipStream_t st,
                 Timing* tm);
int launch_density_gen(a2c_fe_ctx* c, const double* dX);  // fills drho, dFp, demb
int launch_eval_gen(a2c_fe_ctx* c, const double* dX, double* dG, double* dF, bool timed, Timing* tm);
int launch_chem_gen(a2c_fe_ctx* c, const double* dX, const double* coe_h, double gamma_bd, double* dgam,
                    int32_t* dfull, const double* dcorr);
void gen_free(a2c_fe_ctx* c);
int lmvm_minimize(a2c_fe_ctx* c, const double* X0, const a2c_lmvm_opts* o, double* Xout, a2c_lmvm_report* rep);
int launch_chem(a2c_fe_ctx* c, const double* dX, const double* coe_pd, const double* coe_h,
                double gamma_bd, double* dgam, int32_t* dfull, double* dcorr);  // occupancy.hip
// Scratch of one diffusion step: f (n_h doubles), block partials of the
// balance (4 per block of 256 H sites) and the balance itself (4 doubles).
struct DiffuseScratch {
  double* uv;   // 2 nH: (x e^{f/2}, (1-x) e^{-f/2}) per site, f = gamma - ln(x/(1-x)); NaN where |f| >= 700
  double* part;
  double* bal;
};
int diffuse_blocks(int nh);
int launch_diffuse(a2c_fe_ctx* c, double dt, double prefactor, double xLb, double xUb,
                   const double* dgam, const int32_t* dfull, const DiffuseScratch& w, double* dxnew,
                   Timing* tm = nullptr);

// Event timing of individual kernels on the context stream: mark() records
// the next preallocated event; durations are differences of consecutive marks.
struct Timing {
  hipEvent_t* ev = nullptr;
  int cap = 0;
  int n = 0;
  const char* name[8] = {};
  bool on = false;
  void mark(hipStream_t s, const char* nm) {
    if (!on || n >= cap) return;
    if (n < 8) name[n] = nm;
    hipEventRecord(ev[n], s);
    ++n;
  }
};

}  // namespace a2c
