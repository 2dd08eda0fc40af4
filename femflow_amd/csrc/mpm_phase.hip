// Phase kernels on caller-owned dense grids in the reference's layouts:
// grid_v (R+1)^d x d and grid_m (R+1)^d, row-major [i, j(, k)].  These back
// the drop-in phase functions three_d.{p2g,grid_op,g2p} and
// two_d.{p2g,grid_op,g2p} (FP32 or FP64, whichever the caller's arrays are).
// One thread per particle (P2G, G2P) or per node (grid update).  P2G has two
// forms, by size: see p2g_sort_from.
#include <climits>

#include "mpm_cellsum.h"
#include "mpm_math.h"
#include "mpm_phase.h"
#include "mpm_sort.h"
#include "mpm_sort_dev.h"

namespace mpm {

template <typename T> struct PhaseArgs {
  int64_t n;
  int res, quirks, boundary, bound, mat_scalar, kind_override, uniform;
  T inv_dx, dx, dt, vol, gravity, hardening, theta_c, theta_s;
  T mass1, mu1, lam1;  // every particle's, when uniform
  T* x;
  T* v;
  T* F;
  T* C;
  T* Jp;
  const T* mass;
  const T* mu0;
  const T* lam0;
  const int32_t* material;
  T* grid_v;
  T* grid_m;
  unsigned long long* oob;
  int nmat;
  MatParams mats[MPM_PHASE_MAX_MATERIALS];
};

template <typename T>
__device__ __forceinline__ void material_of(const PhaseArgs<T>& a, int64_t p, int& kind, T& h,
                                            T& tc, T& ts) {
  if (a.kind_override >= 0) {
    kind = a.kind_override;
    h = a.hardening;
    tc = a.theta_c;
    ts = a.theta_s;
    return;
  }
  int id = a.material ? a.material[p] : 0;
  id = id < 0 ? 0 : (id >= a.nmat ? a.nmat - 1 : id);
  const MatParams m = a.mats[id];
  kind = m.kind;
  h = (T)m.hardening;
  tc = (T)m.theta_c;
  ts = (T)m.theta_s;
}

template <typename T>
__device__ __forceinline__ void constants_of(const PhaseArgs<T>& a, int64_t p, T& m, T& mu0, T& lam0) {
  if (a.uniform) {
    m = a.mass1;
    mu0 = a.mu1;
    lam0 = a.lam1;
    return;
  }
  const int64_t i = a.mat_scalar ? 0 : p;
  m = a.mass[i];
  mu0 = a.mu0[i];
  lam0 = a.lam0[i];
}

// base = trunc(x inv_dx - 0.5) (three_d/p2g.py:50) with the stencil inside
// [0, R] (utils.py:138-150): valid iff -1 < x inv_dx - 0.5 < R - 1.
template <typename T, int DIM>
__device__ __forceinline__ bool locate(const T* xp, T inv_dx, int res, int base[DIM], T fx[DIM]) {
  bool ok = true;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const T s = xp[d] * inv_dx;
    const T t = fma(xp[d], inv_dx, T(-0.5));  // one rounding in every kernel, so that all agree on who is off the grid
    ok = ok && (t > T(-1)) && (t < T(res - 1));
    base[d] = ok ? (int)t : 0;
    fx[d] = s - (T)base[d];
  }
  return ok;
}

// Adds channel c (momentum, then mass) at node b to the grids.
template <typename T, int DIM>
__device__ __forceinline__ void add_to_grid(const PhaseArgs<T>& a, const int* b, int c, T v) {
  const int64_t r1 = a.res + 1;
  int64_t node = (int64_t)b[0] * r1 + b[1];
  if constexpr (DIM == 3) node = node * r1 + b[2];
  if (c < DIM) atomicAdd(a.grid_v + DIM * node + c, v);
  else atomicAdd(a.grid_m + node, v);
}

// The cell-sum table entry e of particle p; false, with its terms already added
// to the grids, if they are not all finite.
template <typename Sum, typename T, int DIM>
__device__ __forceinline__ bool write_entry(const PhaseArgs<T>& a, int64_t p, const int (&base)[DIM],
                                            const T (&fx)[DIM], T* e) {
  int kind;
  T h, tc, ts;
  material_of(a, p, kind, h, tc, ts);
  T m, mu0, lam0, mu, lam;
  constants_of(a, p, m, mu0, lam0);
  lame<T>(kind, h, mu0, lam0, a.Jp[p], mu, lam);
  const bool textbook = a.quirks == MPM_QUIRKS_TEXTBOOK;
  T A[DIM * DIM];
  if constexpr (DIM == 3)
    affine3<T>(a.F + 9 * p, a.C + 9 * p, m, mu, lam, kind, a.inv_dx, a.dt, a.vol, textbook, A);
  else
    affine2<T>(a.F + 4 * p, a.C + 4 * p, m, mu, lam, kind, a.inv_dx, a.dt, a.vol, textbook, A);
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    T mid = T(0);  // A (n - fx) dx at the middle node
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
      const T ad = A[DIM * d + c] * a.dx;
      e[d * Sum::ROW + 1 + c] = ad;
      mid += ad * (T(1) - fx[c]);
    }
    e[d * Sum::ROW] = m * a.v[DIM * p + d] + mid;
  }
  e[DIM * Sum::ROW] = m;
#pragma unroll
  for (int c = 0; c < DIM; ++c) e[DIM * Sum::ROW + 1 + c] = T(0);
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    T w[3];
    bspline(fx[d], w);
#pragma unroll
    for (int c = 0; c < 3; ++c) e[(DIM + 1) * Sum::ROW + 3 * d + c] = w[c];
  }
  if (Sum::finite(e)) return true;
#pragma unroll
  for (int d = 0; d < DIM; ++d) e[d * Sum::ROW] = m * a.v[DIM * p + d];
  Sum::scatter_one(e, base, fx, [&](const int* b, int c, T v) { add_to_grid<T, DIM>(a, b, c, v); });
  return false;
}

// P2G of few particles (or without scratch memory) in the order in which they
// come.  A workgroup takes THREADS of them, finds the bounding box of their
// stencils, and
// - where neighbouring lanes share cells (cell order, BOX_RUN particles per run and
//   more) or the box has few adds per node, takes the sums of mpm_cellsum.h: in the
//   one case a cell's particles would add to the same LDS words one after the other,
//   in the other an arena would be cleared and read for nothing, and one particle's
//   nodes side by side make better atomics than one lane per particle;
// - else adds particle by particle into an LDS arena over the box, which goes to
//   memory once; layers of the box that the arena cannot hold go to memory particle
//   by particle.
// What bounds it: up to a few thousand particles the chain of loads, stress and
// LDS adds of one workgroup, then the arenas' flushes (each workgroup's box is
// that of the whole body when the order is arbitrary).
// Small workgroups spread few particles over more compute units: 2,048 3D
// particles at 256 / 512 / 1,024 threads 17 / 26 / 46 us at 16 per cell and 23
// / 30 / 47 at 2; in 2D, with a third of the adds, 512 is the best from 8,192
// on (16,384 at 2 per cell 29 / 27 / 26, 8,192 16 / 13 / 15).
// The arena is FP64 for FP32 particles too: LDS adds of floats run at a third
// of a lane per cycle here, those of doubles at about five (8,192 2D FP32
// particles 41 us with an FP32 arena, 9 with this one).
// Per-particle device atomics with sums over runs of lanes, which this replaces /
// always the arena / this, in us: arbitrary order, 8,192 2D FP64 at 16 per cell 30 /
// 7 / 7, 2,048 3D FP64 at 16 55 / 18 / 18, 2,048 3D at 0.05 50 / 57 / 24, 8,192 2D at
// 0.25 15 / 29 / 21, 131,072 3D FP32 at 2 897 / 901 / 304; row-major cell order, 3D
// FP32, 885,000 at 2 / 16 per cell 573, 242 / 331, 484 / 319, 201, 131,072 at 16 57 /
// 65 / 34; 500,000 2D FP32 at 2 / 16 48, 24 / 38, 66 / 39, 36 (one workgroup per
// compute unit: the loads of dense cells in 2D are what the arena's LDS costs).
template <int DIM> constexpr int BOX_THREADS_OF = DIM == 3 ? 256 : 512;
// Particles per run of lanes from which the sums are as fast as the arena: in us
// (arena / sums), 3D FP32 131,072 at 2 / 4 / 8 per cell 70, 57, 54 / 61, 42, 49 and
// 4,000 FP64 at 2 / 8 22, 25 / 23, 19; 2D FP32 80,000 at 2 / 4 / 8 10, 11, 14 / 16, 16, 11.
template <int DIM> constexpr int BOX_RUN_OF = DIM == 3 ? 3 : 6;
constexpr int BOX_WORDS = (144 << 10) / (int)sizeof(double);

template <typename T, int DIM>
__global__ __launch_bounds__(BOX_THREADS_OF<DIM>) void phase_p2g_box_kernel(PhaseArgs<T> a) {
  constexpr int NCH = DIM + 1, THREADS = BOX_THREADS_OF<DIM>, WAVES = THREADS / 64;
  // the arena, or the table and arena of the cell sums
  using Entry = CellSum<T, DIM, NCH>;
  constexpr int TABLE = (int)sizeof(T) * THREADS * Entry::ENTRY;
  using Sum = CellSum<T, DIM, NCH, ((int)sizeof(double) * BOX_WORDS - TABLE) / ((int)sizeof(double) * NCH), THREADS>;
  union BoxShared {
    double arena[BOX_WORDS];
    typename Sum::Shared sum;
  };
  __shared__ __align__(16) BoxShared sh;
  double* const arena = sh.arena;
  __shared__ int box_w[WAVES][2 * DIM], count_w[WAVES], runs_w[WAVES];
  const int t = threadIdx.x;
  const int64_t p0 = (int64_t)blockIdx.x * THREADS + t;
  const bool inrange = p0 < a.n;
  const int64_t p = inrange ? p0 : 0;
  int base[DIM];
  T fx[DIM];
  const bool located = locate<T, DIM>(a.x + p * DIM, a.inv_dx, a.res, base, fx);
  if (inrange && !located && a.oob) atomicAdd(a.oob, 1ull);
  const bool valid = inrange && located;
  {
    // runs of neighbouring lanes in one cell
    bool first = (t & 63) == 0;
    const unsigned long long in = __ballot(valid);
#pragma unroll
    for (int d = 0; d < DIM; ++d) first = __shfl_up(base[d], 1) != base[d] || first;
    const unsigned long long heads = __ballot(valid && (first || !((in >> ((t & 63) - 1)) & 1ull)));
    if ((t & 63) == 0) {
      count_w[t >> 6] = __popcll(in);
      runs_w[t >> 6] = __popcll(heads);
    }
  }
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    int lo = valid ? base[d] : INT_MAX, hi = valid ? base[d] : INT_MIN;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo = min(lo, __shfl_xor(lo, o));
      hi = max(hi, __shfl_xor(hi, o));
    }
    if ((t & 63) == 0) {
      box_w[t >> 6][d] = lo;
      box_w[t >> 6][DIM + d] = hi;
    }
  }
  __syncthreads();
  int low[DIM], ext[DIM];
  int64_t vol = 1;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    int lo = INT_MAX, hi = INT_MIN;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      lo = min(lo, box_w[w][d]);
      hi = max(hi, box_w[w][DIM + d]);
    }
    low[d] = lo;
    ext[d] = lo <= hi ? hi - lo + 3 : 0;
    vol *= ext[d];
  }
  int count = 0, runs = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    count += count_w[w];
    runs += runs_w[w];
  }
  // (sparse: 0.4 adds per node; 16,384 2D FP64 at 0.3 / 0.5 25 / 27 us as sums, 35 /
  // 27 with the arena)
  const bool merge = runs * BOX_RUN_OF<DIM> <= count, sparse = (int64_t)count * Entry::NODES * 5 < 2 * vol;
  if (2 * count > THREADS && (merge || sparse)) {  // (the same in every wave)
    const bool summed =
        valid && write_entry<Sum, T, DIM>(a, p, base, fx, sh.sum.table + t * Sum::ENTRY);
    auto add = [&](const int* b, int c, T v) { add_to_grid<T, DIM>(a, b, c, v); };
    Sum::prepare(sh.sum, base, summed);
    Sum::sum_groups(sh.sum, base, summed, add);
    Sum::flush(sh.sum, add);
    return;
  }
  // the layers of the first axis that the arena holds
  const int64_t layer = ext[0] ? vol / ext[0] * NCH : 1;
  const int held = (int)min((int64_t)ext[0], BOX_WORDS / layer);
  const int words = held * (int)layer;
  for (int e = t; e < words; e += THREADS) arena[e] = 0.0;
  __syncthreads();
  if (valid) {
    T w[DIM][3];
#pragma unroll
    for (int d = 0; d < DIM; ++d) bspline(fx[d], w[d]);
    int kind;
    T h, tc, ts, m, mu0, lam0, mu, lam;
    material_of(a, p, kind, h, tc, ts);
    constants_of(a, p, m, mu0, lam0);
    lame<T>(kind, h, mu0, lam0, a.Jp[p], mu, lam);
    const bool textbook = a.quirks == MPM_QUIRKS_TEXTBOOK;
    T A[DIM * DIM];
    if constexpr (DIM == 3)
      affine3<T>(a.F + 9 * p, a.C + 9 * p, m, mu, lam, kind, a.inv_dx, a.dt, a.vol, textbook, A);
    else
      affine2<T>(a.F + 4 * p, a.C + 4 * p, m, mu, lam, kind, a.inv_dx, a.dt, a.vol, textbook, A);
    T mv[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) mv[d] = a.v[DIM * p + d] * m;
    const int64_t r1 = a.res + 1;
    constexpr int K = DIM == 3 ? 3 : 1;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int o[3] = {i, j, k};
          T dp[DIM], weight = w[0][i] * w[1][j];
          if constexpr (DIM == 3) weight *= w[2][k];
          const bool inside = base[0] + i - low[0] < held;
          uint32_t at = 0;  // (only used inside)
          int64_t node = 0;
#pragma unroll
          for (int d = 0; d < DIM; ++d) {
            dp[d] = (T(o[d]) - fx[d]) * a.dx;
            at = at * (uint32_t)ext[d] + (uint32_t)(base[d] + o[d] - low[d]);
            node = node * r1 + (base[d] + o[d]);
          }
#pragma unroll
          for (int c = 0; c < NCH; ++c) {
            T v = m;
            if (c < DIM) {
              T ad = A[DIM * c] * dp[0];
#pragma unroll
              for (int e = 1; e < DIM; ++e) ad += A[DIM * c + e] * dp[e];
              v = mv[c] + ad;
            }
            v *= weight;
            if (inside) atomicAdd(&arena[at * NCH + c], (double)v);
            else if (c < DIM) atomicAdd(a.grid_v + DIM * node + c, v);
            else atomicAdd(a.grid_m + node, v);
          }
        }
  }
  __syncthreads();
  for (int e = t; e < words; e += THREADS) {
    const T v = (T)arena[e];
    if (v == T(0)) continue;
    const int c = e % NCH;
    int sl = e / NCH;
    int64_t node = 0, stride = 1;
#pragma unroll
    for (int d = DIM - 1; d >= 0; --d) {
      const int q = d > 0 ? sl % ext[d] : sl;
      sl = d > 0 ? sl / ext[d] : 0;
      node += (low[d] + q) * stride;
      stride *= a.res + 1;
    }
    if (c < DIM) atomicAdd(a.grid_v + DIM * node + c, v);
    else atomicAdd(a.grid_m + node, v);
  }
}

// Particles whose stencil leaves the grid.  A launch of its own ahead of a
// phase's kernels lets the host read the count, and raise, while those still
// run: with the count taken inside the phase kernels and read after them, each
// call left the GPU idle for the 20-25 us that the host needs to see the end
// of one call and to launch the next.
template <typename T, int DIM>
__global__ __launch_bounds__(256) void phase_oob_kernel(const T* __restrict__ x, int64_t n, int res, T inv_dx,
                                                        unsigned long long* __restrict__ oob) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int base[DIM];
  T fx[DIM];
  const bool out = p < n && !locate<T, DIM>(x + p * DIM, inv_dx, res, base, fx);
  const unsigned long long m = __ballot(out);
  if (m && (threadIdx.x & 63) == 0) atomicAdd(oob, (unsigned long long)__popcll(m));
}

// Sort keys of the particles' stencil bases: blocks of 4^3 (3D) or 8^2 (2D)
// cells, then the cell inside the block, so that consecutive particles of
// the sorted order share cells and, 256 at a time, a small bounding box.
// Bases off the grid (and NaN) are clamped; the P2G tests them again.
template <typename T, int DIM>
__device__ __forceinline__ uint32_t phase_key(const T* x, int res, T inv_dx) {
  constexpr int SH = DIM == 3 ? 2 : 3, MASK = (1 << SH) - 1;
  const uint32_t nb = (uint32_t)(res + 1 + MASK) >> SH;
  uint32_t blk = 0, cell = 0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const T t = x[d] * inv_dx - T(0.5);
    const int b = !(t > T(0)) ? 0 : (t < T(res) ? (int)t : res);
    blk = blk * nb + (uint32_t)(b >> SH);
    cell = (cell << SH) | (uint32_t)(b & MASK);
  }
  return (blk << 6) | cell;
}

// One sort tile per workgroup, with its histogram of the sort's first digit.
template <typename T, int DIM, int ITEMS>
__global__ __launch_bounds__(RS_THREADS) void phase_keys_kernel(const T* __restrict__ x, int64_t n, int res, T inv_dx,
                                                                uint32_t* __restrict__ keys, int bits,
                                                                uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[RS_MAX_BINS];
  const int64_t base = (int64_t)blockIdx.x * (ITEMS * RS_THREADS);
  T px[ITEMS][DIM];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t i = base + (int64_t)r * RS_THREADS + threadIdx.x, at = i < n ? i : 0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) px[r][d] = x[at * DIM + d];
  }
  uint32_t k[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t i = base + (int64_t)r * RS_THREADS + threadIdx.x;
    k[r] = phase_key<T, DIM>(px[r], res, inv_dx);
    if (i < n) keys[i] = k[r];
  }
  rs_tile_histogram<ITEMS>(k, n, 0, bits, h, hist);
}

// P2G of particles in cell order (perm), summed per cell and workgroup
// before memory (mpm_cellsum.h).  At 131,072 FP64 particles in arbitrary
// order on a 64^3 grid a scatter with device atomics per particle issues 14
// million of them and takes 1,426 us; sort and sums together take about 65 us
// (p2g_sort_from compares it with phase_p2g_box_kernel by size).
template <typename T, int DIM>
__global__ __launch_bounds__(CELLSUM_THREADS) void phase_p2g_sorted_kernel(PhaseArgs<T> a,
                                                                         const uint32_t* __restrict__ perm) {
  using Sum = CellSum<T, DIM, DIM + 1>;
  __shared__ __align__(16) typename Sum::Shared sh;
  const int64_t q = (int64_t)blockIdx.x * CELLSUM_THREADS + threadIdx.x;
  const bool inrange = q < a.n;
  const int64_t p = inrange ? (int64_t)perm[q] : 0;
  int base[DIM];
  T fx[DIM];
  const bool located = locate<T, DIM>(a.x + p * DIM, a.inv_dx, a.res, base, fx);
  if (inrange && !located && a.oob) atomicAdd(a.oob, 1ull);
  bool valid = inrange && located;
  if (valid) valid = write_entry<Sum, T, DIM>(a, p, base, fx, sh.table + threadIdx.x * Sum::ENTRY);
  auto add = [&](const int* b, int c, T v) { add_to_grid<T, DIM>(a, b, c, v); };
  Sum::prepare(sh, base, valid);
  Sum::sum_groups(sh, base, valid, add);
  Sum::flush(sh, add);
}

// three_d/grid_op.py:25-47 and two_d/grid_op.py:13-24, one thread per node.
template <typename T, int DIM>
__global__ void phase_grid_kernel(PhaseArgs<T> a) {
  const int64_t r1 = a.res + 1;
  int64_t total = r1 * r1;
  if (DIM == 3) total *= r1;
  const int64_t node = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= total) return;
  T* g = a.grid_v + DIM * node;
  const T m = a.grid_m[node];
  if constexpr (DIM == 3) {
    const int64_t i = node / (r1 * r1), j = (node / r1) % r1, k = node % r1;
    T v[3] = {g[0], g[1], g[2]};
    if (m > T(0)) {
      const T lim = a.dx * T(0.9) / a.dt;
#pragma unroll
      for (int d = 0; d < 3; ++d) v[d] /= m;
      v[1] += a.dt * a.gravity;
#pragma unroll
      for (int d = 0; d < 3; ++d) v[d] = tmin(tmax(v[d], -lim), lim);
    }
    const int64_t I[3] = {i, j, k};
    if (a.boundary == MPM_BC_REFERENCE) {
#pragma unroll
      for (int d = 0; d < 3; ++d)
        if (I[d] < 1 || I[d] >= a.res - 1) v[d] = T(0);
    } else {
#pragma unroll
      for (int d = 0; d < 3; ++d)
        if (I[d] < a.bound || I[d] > a.res - a.bound) v[0] = v[1] = v[2] = T(0);
    }
    g[0] = v[0];
    g[1] = v[1];
    g[2] = v[2];
  } else {
    if (!(m > T(0))) return;
    const int64_t i = node / r1, j = node % r1;
    T v[2] = {g[0] / m, g[1] / m};
    v[1] += a.dt * a.gravity;
    if (a.boundary == MPM_BC_REFERENCE) {
      const T xs = T(i) / T(a.res), ys = T(j) / T(a.res);
      if (xs < T(0.05) || xs > T(1) - T(0.05) || ys > T(1) - T(0.05)) v[0] = v[1] = T(0);
      if (ys < T(0.05)) v[1] = tmax(T(0), v[1]);
    } else if (i < a.bound || i > a.res - a.bound || j < a.bound || j > a.res - a.bound) {
      v[0] = v[1] = T(0);
    }
    g[0] = v[0];
    g[1] = v[1];
  }
}

// three_d/grid_op.py:50-67 (check_collision_points), one thread per node of
// the dense (R+1)^3 grid; every plane is tested in turn.
struct PlaneSet {
  PlaneDev p[MAX_PLANES];
  int n;
};

template <typename T>
__global__ void phase_planes_kernel(T* __restrict__ gv, int res, PlaneSet ps) {
  const int64_t r1 = res + 1;
  const int64_t node = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= r1 * r1 * r1) return;
  const int i = (int)(node / (r1 * r1)), j = (int)((node / r1) % r1), k = (int)(node % r1);
  bool hit = false;
  for (int q = 0; q < ps.n; ++q) hit = hit || plane_blocks(ps.p[q], i, j, k);
  if (hit) {
    gv[3 * node] = T(0);
    gv[3 * node + 1] = T(0);
    gv[3 * node + 2] = T(0);
  }
}

// A thread loads its stencil's velocities, all in flight together, with its F
// (3D: whole rows of three nodes), before it uses the first: particles in
// arbitrary order touch a line per load, so what bounds it is the address rate
// and the latency of those loads, with two or three waves per SIMD at 2^17
// particles.  131,072 FP64 particles 28.6 -> 22.6 us, 200,001
// FP32 snow 34 -> 27.
template <typename T, int DIM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void phase_g2p_kernel(PhaseArgs<T> a) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.n) return;
  int base[DIM];
  T fx[DIM];
  if (!locate<T, DIM>(a.x + p * DIM, a.inv_dx, a.res, base, fx)) {
    if (a.oob) atomicAdd(a.oob, 1ull);
    return;
  }
  const int64_t r1 = a.res + 1;
  constexpr int ROWS = DIM == 3 ? 9 : 3;
  T g[ROWS][3 * DIM], Fp[DIM * DIM];
#pragma unroll
  for (int q = 0; q < ROWS; ++q) {
    const T* row = a.grid_v;
    if constexpr (DIM == 3) row += 3 * (((int64_t)(base[0] + q / 3) * r1 + (base[1] + q % 3)) * r1 + base[2]);
    else row += 2 * ((int64_t)(base[0] + q) * r1 + base[1]);
#pragma unroll
    for (int e = 0; e < 3 * DIM; ++e) g[q][e] = row[e];
  }
#pragma unroll
  for (int e = 0; e < DIM * DIM; ++e) Fp[e] = a.F[DIM * DIM * p + e];
  T w[DIM][3];
#pragma unroll
  for (int d = 0; d < DIM; ++d) bspline(fx[d], w[d]);
  int kind;
  T h, tc, ts;
  material_of(a, p, kind, h, tc, ts);
  const T c4 = T(4) * a.inv_dx;
  if constexpr (DIM == 3) {
    T v[3] = {0, 0, 0}, C[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const T weight = w[0][i] * w[1][j] * w[2][k];
          const T dp[3] = {T(i) - fx[0], T(j) - fx[1], T(k) - fx[2]};
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const T wg = weight * g[3 * i + j][3 * k + d];
            v[d] += wg;
#pragma unroll
            for (int e = 0; e < 3; ++e) C[3 * d + e] += c4 * (wg * dp[e]);
          }
        }
    T* xp = a.x + 3 * p;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      a.v[3 * p + d] = v[d];
      xp[d] += a.dt * v[d];
    }
    T M[9], Fn[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      M[i] = a.dt * C[i] + ((i % 4 == 0) ? T(1) : T(0));
      a.C[9 * p + i] = C[i];
    }
    matmul3(M, Fp, Fn);
    if (kind == MPM_SNOW) {
      T U[9], s[3], V[9];
      svd3_checked<T>(Fn, U, s, V);
      const T oldJ = det3(Fn);
      const T lo = T(1) - tc, hi = T(1) + ts;
      // rebuild only when a singular value is actually clamped (otherwise
      // U diag(s) V^T is F itself)
      if (s[0] < lo || s[0] > hi || s[1] < lo || s[1] > hi || s[2] < lo || s[2] > hi) {
#pragma unroll
        for (int c = 0; c < 3; ++c) s[c] = tmin(tmax(s[c], lo), hi);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j)
            Fn[3 * i + j] = U[3 * i] * s[0] * V[3 * j] + U[3 * i + 1] * s[1] * V[3 * j + 1] +
                            U[3 * i + 2] * s[2] * V[3 * j + 2];
      }
      const T det = det3(Fn) + T(1e-10);
      a.Jp[p] = tmin(tmax(a.Jp[p] * oldJ / det, T(0.6)), T(20));
    } else if (kind == MPM_WATER) {
      const T c = tcbrt(det3(Fn));
#pragma unroll
      for (int i = 0; i < 9; ++i) Fn[i] = (i % 4 == 0) ? c : T(0);
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) a.F[9 * p + i] = Fn[i];
  } else {
    T v[2] = {0, 0}, C[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const T weight = w[0][i] * w[1][j];
        const T dp[2] = {T(i) - fx[0], T(j) - fx[1]};
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const T wg = weight * g[i][2 * j + d];
          v[d] += wg;
#pragma unroll
          for (int e = 0; e < 2; ++e) C[2 * d + e] += c4 * (wg * dp[e]);
        }
      }
    T* xp = a.x + 2 * p;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      a.v[2 * p + d] = v[d];
      xp[d] += a.dt * v[d];
    }
    const T M[4] = {T(1) + a.dt * C[0], a.dt * C[1], a.dt * C[2], T(1) + a.dt * C[3]};
    T Fn[4] = {M[0] * Fp[0] + M[1] * Fp[2], M[0] * Fp[1] + M[1] * Fp[3], M[2] * Fp[0] + M[3] * Fp[2],
               M[2] * Fp[1] + M[3] * Fp[3]};
#pragma unroll
    for (int i = 0; i < 4; ++i) a.C[4 * p + i] = C[i];
    // two_d/g2p.py:321-330: SVD rebuild and Jp update for every particle.
    // U diag(s) V^T equals F exactly unless a singular value is clamped, so
    // the rebuild (whose rounding would seed spurious stress) only runs then.
    const T oldJ = Fn[0] * Fn[3] - Fn[1] * Fn[2];
    if (kind == MPM_SNOW) {
      T U[4], s[2], V[4];
      svd2<T>(Fn, U, s, V);
      const T lo = T(1) - tc, hi = T(1) + ts;
      if (s[0] < lo || s[0] > hi || s[1] < lo || s[1] > hi) {
        s[0] = tmin(tmax(s[0], lo), hi);
        s[1] = tmin(tmax(s[1], lo), hi);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            Fn[2 * i + j] = U[2 * i] * s[0] * V[2 * j] + U[2 * i + 1] * s[1] * V[2 * j + 1];
      }
    }
    const T det = Fn[0] * Fn[3] - Fn[1] * Fn[2] + T(1e-10);
    a.Jp[p] = tmin(tmax(a.Jp[p] * oldJ / det, T(0.6)), T(20));
#pragma unroll
    for (int i = 0; i < 4; ++i) a.F[4 * p + i] = Fn[i];
  }
}

// ---------------------------------------------------------------- host ----
template <typename T>
static PhaseArgs<T> make_args(const mpm_params* prm, const mpm_particles* p, int kind_override,
                              double hardening, double theta_c, double theta_s,
                              const mpm_material* mats, int nmat, void* gv, void* gm,
                              unsigned long long* oob) {
  PhaseArgs<T> a{};
  a.n = p ? p->n : 0;
  a.res = prm->res;
  a.quirks = prm->quirks;
  a.boundary = prm->boundary;
  a.bound = prm->bound;
  a.inv_dx = (T)prm->inv_dx;
  a.dx = (T)prm->dx;
  a.dt = (T)prm->dt;
  a.vol = (T)prm->volume;
  a.gravity = (T)prm->gravity;
  a.kind_override = kind_override;
  a.hardening = (T)hardening;
  a.theta_c = (T)theta_c;
  a.theta_s = (T)theta_s;
  if (p) {
    a.mat_scalar = p->mat_scalar;
    a.x = (T*)p->x;
    a.v = (T*)p->v;
    a.F = (T*)p->F;
    a.C = (T*)p->C;
    a.Jp = (T*)p->Jp;
    a.mass = (const T*)p->mass;
    a.mu0 = (const T*)p->mu0;
    a.lam0 = (const T*)p->lambda0;
    a.material = p->material;
  }
  a.grid_v = (T*)gv;
  a.grid_m = (T*)gm;
  a.oob = oob;
  a.nmat = nmat > 0 ? nmat : 1;
  for (int i = 0; i < MPM_PHASE_MAX_MATERIALS; ++i) {
    if (mats && i < nmat) {
      a.mats[i].kind = mats[i].kind;
      a.mats[i].hardening = mats[i].hardening;
      a.mats[i].theta_c = mats[i].theta_c;
      a.mats[i].theta_s = mats[i].theta_s;
    } else {
      a.mats[i].kind = MPM_ELASTIC;
      a.mats[i].hardening = 1.0f;
      a.mats[i].theta_c = 2.5e-2f;
      a.mats[i].theta_s = 7.5e-3f;
    }
  }
  return a;
}

static inline unsigned blocks_for(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

// Smallest particle count of the sorted form, which pays for its sort (six
// small launches), where the other pays for its workgroups' boxes.  Measured on
// particles in arbitrary order, box / sorted in us, at 2 and 16 per cell:
//   3D FP64   2,048: 23 / 45, 17 / 38    8,192: 51 / 50, 20 / 41
//            32,768: 193 / 61, 34 / 46   (FP32 226 / 57, 40 / 42)
//           131,072: 772 / 72, 779 / 70
//   2D FP64  16,384: 27 / 41, 10 / 34    32,768: 64 / 41, 15 / 35
//           131,072: 198 / 50, 144 / 49
// Below one per cell the sort finds nothing to merge (0.25 per cell, box / sorted,
// in calls back to back: 3D 4,096 24 / 53, 131,072 279 / 294; 2D 24,576 30 / 54, 65,536
// 59 / 85), but the host cannot tell such a cloud from a body in a corner of its grid.
static int64_t p2g_sort_from(int dim) { return dim == 3 ? 4096 : 24576; }

// Cells of the key space, or 0 when the sorted form does not apply.
static int64_t p2g_key_space(const mpm_params* prm, int64_t n) {
  const int64_t sh = prm->dim == 3 ? 2 : 3, nb = (prm->res + (1 << sh)) >> sh;
  const int64_t keys = nb * nb * (prm->dim == 3 ? nb : 1) * 64;
  return n < (int64_t(1) << 31) && keys <= (int64_t(1) << 32) ? keys : 0;
}

size_t phase_p2g_workspace_bytes(const mpm_params* prm, int64_t n) {
  if (n < p2g_sort_from(prm->dim) || !p2g_key_space(prm, n)) return 0;
  return sizeof(uint32_t) * 2 * (size_t)n + radix_workspace_bytes(n);
}

template <typename T, int DIM>
static void launch_p2g(hipStream_t st, const PhaseArgs<T>& a, int64_t key_space, void* work) {
  if (!work) {
    constexpr int THREADS = BOX_THREADS_OF<DIM>;
    hipLaunchKernelGGL((phase_p2g_box_kernel<T, DIM>), dim3(blocks_for(a.n, THREADS)), dim3(THREADS), 0, st, a);
    return;
  }
  uint32_t* keys = (uint32_t*)work;
  uint32_t *perm, *ws = keys + 2 * a.n;
  const RadixPlan pl = radix_plan(a.n, (uint32_t)(key_space - 1));
#define MPM_KEYS(I)                                                                                                 \
  hipLaunchKernelGGL((phase_keys_kernel<T, DIM, I>), dim3((unsigned)pl.tiles), dim3(RS_THREADS), 0, st, a.x, a.n, \
                     a.res, a.inv_dx, keys, pl.bits, radix_first_hist(ws, a.n))
  if (pl.items == 4) MPM_KEYS(4);
  else if (pl.items == 8) MPM_KEYS(8);
  else MPM_KEYS(16);
#undef MPM_KEYS
  radix_sort(pl, keys, keys, keys + a.n, a.n, ws, true, true, nullptr, &perm, st);
  hipLaunchKernelGGL((phase_p2g_sorted_kernel<T, DIM>), dim3(blocks_for(a.n, CELLSUM_THREADS)),
                     dim3(CELLSUM_THREADS), 0, st, a, perm);
}

template <typename T>
static void set_uniform(PhaseArgs<T>& a, const double* uniform) {
  if (!uniform) return;
  a.uniform = 1;
  a.mass1 = (T)uniform[0];
  a.mu1 = (T)uniform[1];
  a.lam1 = (T)uniform[2];
}

// work: phase_p2g_workspace_bytes() bytes for the sorted form, null for the
// direct one.  uniform: mass, mu0 and lambda0 of every particle (host), or
// null to read them from p.
void phase_p2g(hipStream_t st, const mpm_params* prm, const mpm_particles* p, int kind_override,
               double hardening, const mpm_material* mats, int nmat, void* gv, void* gm,
               unsigned long long* oob, void* work, const double* uniform) {
  if (p->n <= 0) return;
  const int64_t keys = p2g_key_space(prm, p->n);
  if (p->dtype == MPM_F64) {
    auto a = make_args<double>(prm, p, kind_override, hardening, 0, 0, mats, nmat, gv, gm, oob);
    set_uniform(a, uniform);
    if (prm->dim == 3) launch_p2g<double, 3>(st, a, keys, work);
    else launch_p2g<double, 2>(st, a, keys, work);
  } else {
    auto a = make_args<float>(prm, p, kind_override, hardening, 0, 0, mats, nmat, gv, gm, oob);
    set_uniform(a, uniform);
    if (prm->dim == 3) launch_p2g<float, 3>(st, a, keys, work);
    else launch_p2g<float, 2>(st, a, keys, work);
  }
}

void phase_oob(hipStream_t st, const mpm_params* prm, const mpm_particles* p, unsigned long long* oob) {
  if (p->n <= 0) return;
  const unsigned nb = blocks_for(p->n, 256);
#define MPM_OOB(T, D)                                                                                          \
  hipLaunchKernelGGL((phase_oob_kernel<T, D>), dim3(nb), dim3(256), 0, st, (const T*)p->x, p->n, prm->res, \
                     (T)prm->inv_dx, oob)
  if (p->dtype == MPM_F64) {
    if (prm->dim == 3) MPM_OOB(double, 3);
    else MPM_OOB(double, 2);
  } else {
    if (prm->dim == 3) MPM_OOB(float, 3);
    else MPM_OOB(float, 2);
  }
#undef MPM_OOB
}

void phase_grid_op(hipStream_t st, const mpm_params* prm, int dtype, void* gv, const void* gm) {
  const int64_t r1 = prm->res + 1;
  const int64_t total = prm->dim == 3 ? r1 * r1 * r1 : r1 * r1;
  const unsigned nb = blocks_for(total, 256);
  if (dtype == MPM_F64) {
    auto a = make_args<double>(prm, nullptr, -1, 1, 0, 0, nullptr, 0, gv, (void*)gm, nullptr);
    if (prm->dim == 3) hipLaunchKernelGGL((phase_grid_kernel<double, 3>), dim3(nb), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((phase_grid_kernel<double, 2>), dim3(nb), dim3(256), 0, st, a);
  } else {
    auto a = make_args<float>(prm, nullptr, -1, 1, 0, 0, nullptr, 0, gv, (void*)gm, nullptr);
    if (prm->dim == 3) hipLaunchKernelGGL((phase_grid_kernel<float, 3>), dim3(nb), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((phase_grid_kernel<float, 2>), dim3(nb), dim3(256), 0, st, a);
  }
}

void phase_planes(hipStream_t st, int dtype, int res, const PlaneDev* planes, int n, void* gv) {
  PlaneSet ps{};
  for (int q = 0; q < n; ++q) ps.p[q] = planes[q];
  ps.n = n;
  const int64_t r1 = res + 1;
  const unsigned nb = blocks_for(r1 * r1 * r1, 256);
  if (dtype == MPM_F64) hipLaunchKernelGGL(phase_planes_kernel<double>, dim3(nb), dim3(256), 0, st, (double*)gv, res, ps);
  else hipLaunchKernelGGL(phase_planes_kernel<float>, dim3(nb), dim3(256), 0, st, (float*)gv, res, ps);
}

void phase_g2p(hipStream_t st, const mpm_params* prm, mpm_particles* p, int kind_override,
               double theta_c, double theta_s, const mpm_material* mats, int nmat, const void* gv,
               unsigned long long* oob) {
  if (p->n <= 0) return;
  const unsigned nb = blocks_for(p->n, 256);
  if (p->dtype == MPM_F64) {
    auto a = make_args<double>(prm, p, kind_override, 1, theta_c, theta_s, mats, nmat, (void*)gv,
                               nullptr, oob);
    if (prm->dim == 3) hipLaunchKernelGGL((phase_g2p_kernel<double, 3>), dim3(nb), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((phase_g2p_kernel<double, 2>), dim3(nb), dim3(256), 0, st, a);
  } else {
    auto a = make_args<float>(prm, p, kind_override, 1, theta_c, theta_s, mats, nmat, (void*)gv,
                              nullptr, oob);
    if (prm->dim == 3) hipLaunchKernelGGL((phase_g2p_kernel<float, 3>), dim3(nb), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((phase_g2p_kernel<float, 2>), dim3(nb), dim3(256), 0, st, a);
  }
}

}  // namespace mpm
