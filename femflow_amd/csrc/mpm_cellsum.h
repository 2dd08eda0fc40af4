// Particle-to-node sums without one atomic per particle and node.
//
// A workgroup takes THREADS consecutive particles of a cell-ordered
// list.  Each thread writes its particle's B-spline weights and linear terms
// to an LDS table; each wave then walks the groups of equal stencil bases
// among its 64 particles with one lane per (node, channel) output (3D: 54
// lanes with up to two channels each; 2D: two sets of 27 lanes that take
// alternate particles), so a group of m particles ends in one add per output
// instead of m.  The adds go to an LDS
// arena over the workgroup's stencil bounding box, which is added to memory
// once, one device atomic per nonzero value.  Device-scope float atomics run
// at about 1e10 per second over the whole chip here (one L2 per XCD, so they
// are served behind it), which is what a per-particle scatter is bound by.
//
// Value of channel c at stencil node (i, j[, k]) of a particle:
//   w_i w_j [w_k] (q[c] + A[c][0] (i - 1) + A[c][1] (j - 1) [+ A[c][2] (k - 1)]),
// q being the value at the middle node: expanded there, the terms are no larger
// than those of A (n - fx) and round no more (about node 0 the offset A fx and
// what it takes back are up to three times as large).
#pragma once
#include <hip/hip_runtime.h>

#include <climits>

#include "mpm_math.h"

namespace mpm {

constexpr int CELLSUM_THREADS = 256;

// ARENA: nodes of the LDS arena; a workgroup whose box is larger adds each
// group's sums to memory.  FP64 for FP32 particles too, since LDS adds of floats
// run at a third of a lane per cycle and those of doubles at about five (131,072
// FP32 particles, sort included, 80 -> 65 us at 2 per cell and 83 -> 64 at 16, with
// an arena of 1,024 FP32 nodes before).  576 leaves room for two workgroups of the
// phase P2G (FP64, 3D) per compute unit, whose particles come in blocks of cells.
template <typename T, int DIM, int NCH, int ARENA = 576, int THREADS = CELLSUM_THREADS> struct CellSum {
  static constexpr int NODES = DIM == 3 ? 27 : 9;
  static constexpr int ROW = DIM == 3 ? 4 : 3;  // q, A[0..DIM-1] of a channel
  // per-particle table entry: NCH rows, then DIM x 3 weights, padded to 16
  // bytes, so that a 3D row is read 16 bytes at a time
  static constexpr int PAD = 16 / (int)sizeof(T);
  static constexpr int ENTRY = (NCH * ROW + 3 * DIM + PAD - 1) / PAD * PAD;
  typedef T Row3 __attribute__((ext_vector_type(4), aligned(16)));
  struct alignas(16) Shared {
    T table[THREADS * ENTRY];
    double arena[ARENA * NCH];
    int box_w[THREADS / 64][2 * DIM];
    int box[2 * DIM];  // low corner, extent (0: the box does not fit the arena)
  };

  // Whether all linear terms of a table entry are finite.  sum_groups must not see
  // others: q + A (n - 1) is A (n - fx) multiplied out, where an infinite A gives
  // NaN for an infinity.
  static __device__ __forceinline__ bool finite(const T* e) {
    T zero = T(0);
#pragma unroll
    for (int r = 0; r < NCH * ROW; ++r) zero += e[r] * T(0);
    return zero == T(0);
  }

  // One particle's terms to its nodes, for an entry whose q is the value at fx
  // (without A fx taken off).  Rolled: it is rarely run.
  template <typename Add>
  static __device__ __forceinline__ void scatter_one(const T* e, const int (&base)[DIM], const T (&fx)[DIM], Add add) {
#pragma unroll 1
    for (int node = 0; node < NODES; ++node) {
      int o[DIM], b[DIM], rest = node;
      T w = T(1);
#pragma unroll
      for (int d = DIM - 1; d >= 0; --d) {
        o[d] = rest % 3;
        rest /= 3;
        b[d] = base[d] + o[d];
      }
#pragma unroll
      for (int d = 0; d < DIM; ++d) w *= e[NCH * ROW + 3 * d + o[d]];
#pragma unroll 1
      for (int c = 0; c < NCH; ++c) {
        T ad = T(0);
#pragma unroll
        for (int d = 0; d < DIM; ++d) ad += e[c * ROW + 1 + d] * (T(o[d]) - fx[d]);
        add(b, c, w * (e[c * ROW] + ad));
      }
    }
  }

  // Bounding box of the workgroup's stencils (valid particles) and the
  // cleared arena.  Every thread of the workgroup calls it; ends in a
  // barrier, so the table may be written before it and read after it.
  static __device__ __forceinline__ void prepare(Shared& sh, const int (&base)[DIM], bool valid) {
    const int t = threadIdx.x;
    int lo[DIM], hi[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      lo[d] = valid ? base[d] : INT_MAX;
      hi[d] = valid ? base[d] : INT_MIN;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        lo[d] = min(lo[d], __shfl_xor(lo[d], o));
        hi[d] = max(hi[d], __shfl_xor(hi[d], o));
      }
      if ((t & 63) == 0) {
        sh.box_w[t >> 6][d] = lo[d];
        sh.box_w[t >> 6][DIM + d] = hi[d];
      }
    }
    __syncthreads();
    if (t == 0) {
      int64_t vol = 1;
      int l[DIM], e[DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        int a = INT_MAX, b = INT_MIN;
        for (int w = 0; w < THREADS / 64; ++w) {
          a = min(a, sh.box_w[w][d]);
          b = max(b, sh.box_w[w][DIM + d]);
        }
        l[d] = a;
        e[d] = a <= b ? b - a + 3 : 0;
        vol *= e[d];
      }
      const bool fits = vol > 0 && vol <= ARENA;
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        sh.box[d] = l[d];
        sh.box[DIM + d] = fits ? e[d] : 0;
      }
    }
    __syncthreads();
    const int n = volume(sh) * NCH;
    for (int e = t; e < n; e += THREADS) sh.arena[e] = 0.0;
    __syncthreads();
  }

  static __device__ __forceinline__ int volume(const Shared& sh) {
    int v = 1;
#pragma unroll
    for (int d = 0; d < DIM; ++d) v *= sh.box[DIM + d];
    return v;
  }

  // Sums every group of this wave's particles that share a base (the lanes
  // of a group need not be neighbours: an order that was by cell some
  // substeps ago serves as well).  direct(node, channel, value) adds to
  // memory where the box does not fit the arena.  The table entries of the
  // wave were written by its own lanes; prepare()'s barriers order them.
  template <typename Add>
  static __device__ __forceinline__ void sum_groups(Shared& sh, const int (&base)[DIM], bool valid, Add direct) {
    const int t = threadIdx.x, lane = t & 63;
    unsigned long long left = __ballot(valid);
    constexpr int OUT = DIM == 3 ? 27 : NODES * NCH;
    const int sub = lane / OUT, o = lane - sub * OUT;  // sub 2: idle lanes
    const int node = DIM == 3 ? o : o % NODES;
    const int i = DIM == 3 ? node / 9 : node / 3, j = DIM == 3 ? (node / 3) % 3 : node % 3, k = node % 3;
    const int c0 = DIM == 3 ? 2 * sub : o / NODES;
    const bool on0 = lane < 2 * OUT && c0 < NCH, on1 = DIM == 3 && lane < OUT * 2 && c0 + 1 < NCH;
    const T fi = (T)(i - 1), fj = (T)(j - 1), fk = (T)(k - 1);
    const int r0 = (on0 ? c0 : 0) * ROW, r1 = (on1 ? c0 + 1 : 0) * ROW;
    const int wi = NCH * ROW + i, wj = NCH * ROW + 3 + j, wk = NCH * ROW + (DIM == 3 ? 6 + k : 0);
    const bool arena = sh.box[DIM] > 0;
    while (left) {
      const int s = __builtin_ctzll(left);
      int b[DIM];
      bool same = valid;
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        b[d] = __builtin_amdgcn_readlane(base[d], s);
        same = same && base[d] == b[d];
      }
      unsigned long long m = __ballot(same);
      left &= ~m;
      // FP64 also over the group: its members' terms are of one size, and in
      // dense cells FP32 sums of them were most of the error
      double a0 = 0.0, a1 = 0.0;
      const T* wave = sh.table + (t & ~63) * ENTRY;
      if constexpr (DIM == 3) {
#pragma unroll 2
        while (m) {
          const T* tab = wave + __builtin_ctzll(m) * ENTRY;
          m &= m - 1;
          const T w = tab[wi] * tab[wj] * tab[wk];
          const Row3 q0 = *reinterpret_cast<const Row3*>(tab + r0), q1 = *reinterpret_cast<const Row3*>(tab + r1);
          a0 += (double)(w * (q0.x + q0.y * fi + q0.z * fj + q0.w * fk));
          a1 += (double)(w * (q1.x + q1.y * fi + q1.z * fj + q1.w * fk));
        }
      } else {
        while (m) {  // two particles at a time, one per group of lanes
          const int p0 = __builtin_ctzll(m);
          m &= m - 1;
          const int p1 = m ? __builtin_ctzll(m) : -1;
          m &= m - 1;
          const int p = sub == 0 ? p0 : p1;
          const T* tab = wave + (p < 0 ? p0 : p) * ENTRY;
          const T v = tab[wi] * tab[wj] * (tab[r0] + tab[r0 + 1] * fi + tab[r0 + 2] * fj);
          a0 += (double)(p < 0 ? T(0) : v);
        }
      }
      if (arena) {
        int at = (b[0] + i - sh.box[0]) * sh.box[DIM + 1] + (b[1] + j - sh.box[1]);
        if constexpr (DIM == 3) at = at * sh.box[DIM + 2] + (b[2] + k - sh.box[2]);
        if (on0) atomicAdd(&sh.arena[at * NCH + c0], a0);
        if (on1) atomicAdd(&sh.arena[at * NCH + c0 + 1], a1);
      } else {
        b[0] += i;
        b[1] += j;
        if constexpr (DIM == 3) b[2] += k;
        if (on0) direct(b, c0, (T)a0);
        if (on1) direct(b, c0 + 1, (T)a1);
      }
    }
  }

  // After every wave's sum_groups: the arena's nonzero values to memory.
  template <typename Add> static __device__ __forceinline__ void flush(Shared& sh, Add add) {
    __syncthreads();
    const int n = volume(sh) * NCH;
    for (int e = threadIdx.x; e < n; e += THREADS) {
      const T v = (T)sh.arena[e];
      if (v != T(0)) {
        const int c = e % NCH;
        int sl = e / NCH;
        int b[DIM];
#pragma unroll
        for (int d = DIM - 1; d > 0; --d) {
          b[d] = sh.box[d] + sl % sh.box[DIM + d];
          sl /= sh.box[DIM + d];
        }
        b[0] = sh.box[0] + sl;
        add(b, c, v);
      }
    }
  }
};

}  // namespace mpm
