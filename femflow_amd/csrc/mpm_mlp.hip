// BF16 MFMA training and inference kernels of the grid-corrector MLP.
//
// mlp_forward_kernel   X -> H1 -> H2 -> Y in one pass over the rows
// mlp_dgrad_kernel     dY -> dH2 -> dH1 in one pass over the rows
// mlp_wgrad_kernel     the weight and bias gradients, split over the rows
// mlp_reduce_kernel    sums the splits into the gradient
// Operands are BF16 (uint16 storage), accumulation FP32 on
// v_mfma_f32_16x16x32_bf16.
//
// At 32,768 rows one kernel per layer took 980 us for 60 MB and 13 GFLOP:
// loads behind a bounds test each waited for the one before (a lane mask per
// load; forward and dH 215 us), the bias sums ran on a few dozen workgroups
// (588 us), and the weight gradients gathered both operands two bytes at a
// time and ended in a million device atomics (184 us).  Now: forward 17 us,
// dH 13 us, weight and bias gradients 28 + 6 us.
#include <hip/hip_runtime.h>

#include "mpm_mlp.h"

namespace mpm {

constexpr int ROW_WAVES = 8, MLP_TILE = 16 * ROW_WAVES;  // rows per workgroup and turn of the row passes
constexpr int HSTR = MLP_H + 8;                          // LDS row stride of an activation tile

// Weights in LDS in the order of the MFMA operands: the 16 bytes of lane l for
// columns 16 u .. of step k0 / 32 sit at ((k0 / 32) * (N / 16) + u) * 64 + l,
// so that a wave reads 1 KB in a row.
template <int N, int K>
__device__ __forceinline__ void load_weights(uint4* lds, const uint16_t* __restrict__ B) {
  constexpr int PIECES = N * K / 8;
#pragma unroll 4
  for (int e = threadIdx.x; e < PIECES; e += 64 * ROW_WAVES) {
    const int r = e / (K / 8), c = e % (K / 8);
    lds[((c >> 2) * (N / 16) + (r >> 4)) * 64 + (c & 3) * 16 + (r & 15)] =
        *reinterpret_cast<const uint4*>(B + (size_t)e * 8);
  }
}

// acc[u] (16 rows x 128 columns of one wave) += A B^T, one operand a[] per 32
// of K, B from load_weights.
template <int STEPS>
__device__ __forceinline__ void mlp_layer(const uint4 (&a)[STEPS], const uint4* B, int lane, floatx4 (&acc)[8]) {
#pragma unroll
  for (int k = 0; k < STEPS; ++k)
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] = mfma16x16x32(a[k], B[(k * 8 + u) * 64 + lane], acc[u]);
}

template <int STEPS> __device__ __forceinline__ void load_rows(const uint16_t* row, uint4 (&a)[STEPS]) {
#pragma unroll
  for (int k = 0; k < STEPS; ++k) a[k] = *reinterpret_cast<const uint4*>(row + 32 * k);
}

// Orders a wave's own LDS writes and reads (its lanes read each other's).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ void zero_acc(floatx4 (&acc)[8]) {
#pragma unroll
  for (int u = 0; u < 8; ++u) acc[u] = floatx4{0.f, 0.f, 0.f, 0.f};
}

// A wave's 16 x 128 BF16 tile between LDS (row stride HSTR) and memory, 16
// bytes per lane, four 256-byte rows per round; rows past M are not touched
// (reads clamp to the last row).
__device__ __forceinline__ void tile_store(const uint16_t* tile, uint16_t* __restrict__ out, int64_t row0, int64_t M,
                                           int lane) {
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int r = it * 4 + (lane >> 4), c = (lane & 15) * 8;
    if (row0 + r < M)
      *reinterpret_cast<uint4*>(out + (row0 + r) * MLP_H + c) = *reinterpret_cast<const uint4*>(tile + r * HSTR + c);
  }
}
__device__ __forceinline__ void tile_load(uint16_t* tile, const uint16_t* __restrict__ in, int64_t row0, int64_t M,
                                          int lane) {
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int r = it * 4 + (lane >> 4), c = (lane & 15) * 8;
    const int64_t row = row0 + r < M ? row0 + r : M - 1;
    *reinterpret_cast<uint4*>(tile + r * HSTR + c) = *reinterpret_cast<const uint4*>(in + row * MLP_H + c);
  }
}

// tile[r][col] = relu(acc + bias)
__device__ __forceinline__ void relu_tile(const floatx4 (&acc)[8], const float* __restrict__ bias, uint16_t* tile,
                                          int lane) {
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int col = 16 * u + (lane & 15);
    const float bb = bias[col];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = acc[u][r] + bb;
      tile[((lane >> 4) * 4 + r) * HSTR + col] = f2bf(v > 0.f ? v : 0.f);
    }
  }
}

// A workgroup keeps all weights in LDS (124 KB) and takes 128 rows at a time,
// 16 per wave: three layers, the hidden activations through the wave's LDS
// tile (and to memory for the backward pass).  A wave's rows of X are in
// flight while the weights are copied, and the next turn's while this one's
// layers run.  What bounds it: one turn's chain of loads, products and
// stores, at 32,768 rows one turn of every compute unit: 17 us.  With the
// weights read from L2 by every wave (250 MB of them) it took 28.
struct ForwardShared {
  uint4 w1[MLP_H * MLP_INP / 8], w2[MLP_H * MLP_H / 8], w3[MLP_OUTP * MLP_H / 8];
  uint16_t tile[ROW_WAVES][16 * HSTR];
};
__global__ __launch_bounds__(64 * ROW_WAVES) void mlp_forward_kernel(const uint16_t* __restrict__ K,
                                                                     const float* __restrict__ P,
                                                                     const uint16_t* __restrict__ X, int64_t M,
                                                                     uint16_t* __restrict__ H1,
                                                                     uint16_t* __restrict__ H2,
                                                                     float* __restrict__ Y) {
  __shared__ __align__(16) ForwardShared sh;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int li = lane & 15, lk = (lane >> 4) * 8;
  uint16_t* const tile = sh.tile[wv];
  const int64_t turn = (int64_t)gridDim.x * MLP_TILE;
  int64_t row0 = (int64_t)blockIdx.x * MLP_TILE + wv * 16;
  auto x_row = [&](int64_t r0) { return X + (r0 + li < M ? r0 + li : M - 1) * MLP_INP + lk; };
  uint4 x[MLP_INP / 32];
  load_rows(x_row(row0), x);
  load_weights<MLP_H, MLP_INP>(sh.w1, K + K_W1);
  load_weights<MLP_H, MLP_H>(sh.w2, K + K_W2);
  load_weights<MLP_OUTP, MLP_H>(sh.w3, K + K_W3);
  __syncthreads();
  for (; row0 < M; row0 += turn) {
    floatx4 acc[8];
    uint4 h[MLP_H / 32];
    zero_acc(acc);
    mlp_layer(x, sh.w1, lane, acc);
    if (row0 + turn < M) load_rows(x_row(row0 + turn), x);
    relu_tile(acc, P + P_B1, tile, lane);
    wave_fence();
    load_rows(tile + li * HSTR + lk, h);
    tile_store(tile, H1, row0, M, lane);
    wave_fence();
    zero_acc(acc);
    mlp_layer(h, sh.w2, lane, acc);
    relu_tile(acc, P + P_B2, tile, lane);
    wave_fence();
    load_rows(tile + li * HSTR + lk, h);
    tile_store(tile, H2, row0, M, lane);
    wave_fence();
    floatx4 y = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < MLP_H / 32; ++k) y = mfma16x16x32(h[k], sh.w3[k * 64 + lane], y);
    if (li < MLP_OUT) {
      const float bb = P[P_B3 + li];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = row0 + (lane >> 4) * 4 + r;
        if (row < M) Y[row * MLP_OUTP + li] = y[r] + bb;
      }
    }
  }
}

// tile[r][col] = acc where the activation in `tile` is positive, else 0
__device__ __forceinline__ void mask_tile(const floatx4 (&acc)[8], uint16_t* tile, int lane) {
#pragma unroll
  for (int u = 0; u < 8; ++u)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      uint16_t* h = tile + ((lane >> 4) * 4 + r) * HSTR + 16 * u + (lane & 15);
      *h = f2bf(bf2f(*h) > 0.f ? acc[u][r] : 0.f);
    }
}

// dH2 = (dY W3) where H2 > 0, dH1 = (dH2 W2) where H1 > 0, by the forward's
// scheme (32,768 rows 17 -> 13 us).
struct DGradShared {
  uint4 w3t[MLP_H * MLP_DYP / 8], w2t[MLP_H * MLP_H / 8];
  uint16_t tile[2][ROW_WAVES][16 * HSTR];
};
__global__ __launch_bounds__(64 * ROW_WAVES) void mlp_dgrad_kernel(const uint16_t* __restrict__ K, int64_t M,
                                                                   const uint16_t* __restrict__ H1,
                                                                   const uint16_t* __restrict__ H2,
                                                                   const uint16_t* __restrict__ dY,
                                                                   uint16_t* __restrict__ dH2,
                                                                   uint16_t* __restrict__ dH1) {
  __shared__ __align__(16) DGradShared sh;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int li = lane & 15, lk = (lane >> 4) * 8;
  uint16_t *const t1 = sh.tile[0][wv], *const t2 = sh.tile[1][wv];
  const int64_t turn = (int64_t)gridDim.x * MLP_TILE;
  const int64_t first = (int64_t)blockIdx.x * MLP_TILE + wv * 16;
  uint4 y[1], h[MLP_H / 32];
  auto fetch = [&](int64_t row0) {
    load_rows(dY + (row0 + li < M ? row0 + li : M - 1) * MLP_DYP + lk, y);
    tile_load(t2, H2, row0, M, lane);
    tile_load(t1, H1, row0, M, lane);
  };
  load_weights<MLP_H, MLP_DYP>(sh.w3t, K + K_W3T);
  load_weights<MLP_H, MLP_H>(sh.w2t, K + K_W2T);
  if (first < M) fetch(first);
  __syncthreads();
  for (int64_t row0 = first; row0 < M; row0 += turn) {
    if (row0 != first) fetch(row0);
    wave_fence();
    floatx4 acc[8];
    zero_acc(acc);
    mlp_layer(y, sh.w3t, lane, acc);
    mask_tile(acc, t2, lane);
    wave_fence();
    load_rows(t2 + li * HSTR + lk, h);
    tile_store(t2, dH2, row0, M, lane);
    zero_acc(acc);
    mlp_layer(h, sh.w2t, lane, acc);
    mask_tile(acc, t1, lane);
    wave_fence();
    tile_store(t1, dH1, row0, M, lane);
    wave_fence();
  }
}

// ------------------------------------------------------ weight gradients ----
// gW = dH^T In, a product over the rows.  Both operands are row-major with
// the rows as the reduction index, so a lane needs eight rows of one column
// per MFMA operand.  A lane loads eight (or four) columns of each of eight
// rows and transposes the values in registers (one v_perm per pair), which
// gives the operands of eight (four) tiles at once: tile t of lane li stands
// for column 8 li + t (4 li + t).  A wave then has a 128 x 64 block of the
// gradient in its accumulators, 32 products per 32 rows for 16 loads.
// What bounds it is the latency of those loads against the few products they
// feed.  With 128 x 128 blocks a wave took all 512 registers of a SIMD and
// nothing ran while it waited: 38 us at 32,768 rows, 28 with half the block,
// which leaves room for a second wave.  Of those 28, 16 do not depend on the
// rows: launch, the first loads, the sums over waves and the partial gradients.
template <typename V>
__device__ __forceinline__ void load_columns(const uint16_t* __restrict__ src, int64_t ld, int64_t k, int64_t kend,
                                             bool on, V (&raw)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int64_t r = k + j < kend ? k + j : kend - 1;
    raw[j] = *reinterpret_cast<const V*>(src + r * ld);
    if (!on || k + j >= kend) raw[j] = V{};
  }
}
template <typename V, int T> __device__ __forceinline__ void transpose8(const V (&raw)[8], uint4 (&frag)[T]) {
  static_assert(sizeof(V) == 2 * T, "one column per tile");
  uint32_t f[T][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t lo[T / 2], hi[T / 2];
    __builtin_memcpy(lo, &raw[2 * q], sizeof(V));
    __builtin_memcpy(hi, &raw[2 * q + 1], sizeof(V));
#pragma unroll
    for (int c = 0; c < T / 2; ++c) {
      f[2 * c][q] = __builtin_amdgcn_perm(hi[c], lo[c], 0x05040100u);
      f[2 * c + 1][q] = __builtin_amdgcn_perm(hi[c], lo[c], 0x07060302u);
    }
  }
#pragma unroll
  for (int t = 0; t < T; ++t) frag[t] = make_uint4(f[t][0], f[t][1], f[t][2], f[t][3]);
}

constexpr uint32_t BF_ONES = 0x3f803f80u;

struct WGradArgs {
  int64_t M, per;  // rows, rows per workgroup (a multiple of 128)
  const uint16_t *X, *H1, *H2, *dY, *dH2, *dH1;
  float* out;     // one gradient per split, or the gradient itself
  int atomic;     // add to `out` (one array) instead of storing a split's own
};

// Workgroup (split s, job): jobs 0..5 columns 64 job .. of gW1 (column 351,
// which holds no feature, is taken as 1 and gives the bias gradient), jobs 6
// and 7 the halves of gW2, job 8 gW3, gb3 and gb2.  Its four waves take a
// quarter of the split's rows each and add up through LDS.
constexpr int WG_JOBS = 9;
__global__ __launch_bounds__(256, 2) void mlp_wgrad_kernel(WGradArgs g) {
  // two waves' blocks (jobs 0..7), or four waves' 17 tiles (job 8)
  constexpr int SUM_TILES = 4 * 17;
  __shared__ __align__(16) floatx4 sum_s[SUM_TILES][64];
  static_assert(SUM_TILES >= 2 * 32 && SUM_TILES * 64 * 4 >= 128 * 65, "LDS of the three uses");
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int li = lane & 15, grp = lane >> 4;
  // each XCD (workgroup id mod 8) takes a contiguous run of (split, job), jobs
  // fastest, so that a split's nine jobs read its rows through one L2
  const uint32_t xcd = blockIdx.x & 7u, run = gridDim.x >> 3, rem = gridDim.x & 7u;
  const uint32_t at = xcd * run + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
  const int job = (int)(at % WG_JOBS);
  const int64_t split = at / WG_JOBS, r0 = split * g.per;
  const int64_t quarter = g.per / 4;
  const int64_t kb = r0 + wv * quarter;
  const int64_t ke = kb + quarter < g.M ? kb + quarter : g.M;
  float* const out = g.out + (g.atomic ? 0 : split * P_COUNT);
  auto put = [&](int i, float v) {
    if (g.atomic) atomicAdd(out + i, v);
    else out[i] = v;
  };
  if (job < 8) {
    const int col0 = job < 6 ? 64 * job : 64 * (job - 6);
    const uint16_t* A = (job < 6 ? g.dH1 : g.dH2) + 8 * li;
    const uint16_t* B = job < 6 ? g.X : g.H1;
    const int64_t ldb = job < 6 ? MLP_INP : MLP_H;
    const int bc = col0 + 4 * li;
    const bool on = bc < ldb;
    B += on ? bc : 0;
    const bool ones = job == 5 && bc == MLP_IN - 3;  // this lane's tile 3 is column 351
    floatx4 acc[8][4];
#pragma unroll
    for (int ta = 0; ta < 8; ++ta)
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) acc[ta][tb] = floatx4{0.f, 0.f, 0.f, 0.f};
    uint4 ra[8];
    uint2 rb[8];
    if (kb < ke) {
      load_columns(A, MLP_H, kb + 8 * grp, ke, true, ra);
      load_columns(B, ldb, kb + 8 * grp, ke, on, rb);
    }
    for (int64_t k = kb; k < ke; k += 32) {
      uint4 fa[8], fb[4];
      transpose8(ra, fa);
      transpose8(rb, fb);
      if (ones) fb[3] = make_uint4(BF_ONES, BF_ONES, BF_ONES, BF_ONES);
      if (k + 32 < ke) {
        load_columns(A, MLP_H, k + 32 + 8 * grp, ke, true, ra);
        load_columns(B, ldb, k + 32 + 8 * grp, ke, on, rb);
      }
#pragma unroll
      for (int ta = 0; ta < 8; ++ta)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) acc[ta][tb] = mfma16x16x32(fa[ta], fb[tb], acc[ta][tb]);
    }
    // waves 2, 3 -> 0, 1; wave 1 -> 0
#pragma unroll
    for (int half = 2; half >= 1; half >>= 1) {
      if (wv >= half && wv < 2 * half) {
#pragma unroll
        for (int ta = 0; ta < 8; ++ta)
#pragma unroll
          for (int tb = 0; tb < 4; ++tb) sum_s[(wv - half) * 32 + ta * 4 + tb][lane] = acc[ta][tb];
      }
      __syncthreads();
      if (wv < half) {
#pragma unroll
        for (int ta = 0; ta < 8; ++ta)
#pragma unroll
          for (int tb = 0; tb < 4; ++tb) acc[ta][tb] += sum_s[wv * 32 + ta * 4 + tb][lane];
      }
      __syncthreads();
    }
    float* nat = reinterpret_cast<float*>(sum_s);  // [128][65]
    if (wv == 0) {
#pragma unroll
      for (int ta = 0; ta < 8; ++ta)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb)
#pragma unroll
          for (int r = 0; r < 4; ++r) nat[(8 * (grp * 4 + r) + ta) * 65 + 4 * li + tb] = acc[ta][tb][r];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 128 * 64; e += 256) {
      const int m = e >> 6, n = col0 + (e & 63);
      const float v = nat[m * 65 + (e & 63)];
      if (job >= 6) put(P_W2 + m * MLP_H + n, v);
      else if (n < MLP_IN) put(P_W1 + m * MLP_IN + n, v);
      else if (n == MLP_IN) put(P_B1 + m, v);
    }
    return;
  }
  // job 8: A = dY (three columns) with B = H2 and 1; A = dH2 with B = 1
  floatx4 w3[8], b2[8], b3 = floatx4{0.f, 0.f, 0.f, 0.f};
  zero_acc(w3);
  zero_acc(b2);
  const uint4 one = make_uint4(BF_ONES, BF_ONES, BF_ONES, BF_ONES);
  for (int64_t k = kb; k < ke; k += 32) {
    uint4 rh[8], rd[8], fh[8], fd[8];
    load_columns(g.H2 + 8 * li, MLP_H, k + 8 * grp, ke, true, rh);
    load_columns(g.dH2 + 8 * li, MLP_H, k + 8 * grp, ke, true, rd);
    uint32_t y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t r = k + 8 * grp + j;
      y[j] = g.dY[(r < ke ? r : ke - 1) * MLP_DYP + (li < MLP_OUT ? li : 0)];
      if (r >= ke || li >= MLP_OUT) y[j] = 0u;
    }
    transpose8(rh, fh);
    transpose8(rd, fd);
    const uint4 fy = make_uint4(y[0] | (y[1] << 16), y[2] | (y[3] << 16), y[4] | (y[5] << 16), y[6] | (y[7] << 16));
    b3 = mfma16x16x32(fy, one, b3);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      w3[t] = mfma16x16x32(fy, fh[t], w3[t]);
      b2[t] = mfma16x16x32(fd[t], one, b2[t]);
    }
  }
  floatx4(*part)[17][64] = reinterpret_cast<floatx4(*)[17][64]>(sum_s);
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    part[wv][t][lane] = w3[t];
    part[wv][8 + t][lane] = b2[t];
  }
  part[wv][16][lane] = b3;
  __syncthreads();
  if (wv == 0) {
    auto total = [&](int t) { return (part[0][t][lane] + part[1][t][lane]) + (part[2][t][lane] + part[3][t][lane]); };
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const floatx4 w = total(t), b = total(8 + t);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = grp * 4 + r;
        if (m < MLP_OUT) put(P_W3 + m * MLP_H + 8 * li + t, w[r]);
        if (li == 0) put(P_B2 + 8 * m + t, b[r]);
      }
    }
    const floatx4 b = total(16);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (li == 0 && grp * 4 + r < MLP_OUT) put(P_B3 + grp * 4 + r, b[r]);
  }
}

// G += the sum of the splits' gradients, in FP64: with FP32 sums their
// rounding was most of the gradient's error (1.1e-7 of its norm against the
// exact sums at 32,768 rows).
__global__ __launch_bounds__(256) void mlp_reduce_kernel(const float* __restrict__ part, int splits,
                                                         float* __restrict__ G) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P_COUNT) return;
  double s = G[i];
#pragma unroll 16
  for (int k = 0; k < splits; ++k) s += (double)part[(int64_t)k * P_COUNT + i];
  G[i] = (float)s;
}

// Weighted mean squared error of the 3 outputs; writes dL/dY (BF16, ld 32,
// zero padding) and adds the loss to *loss.
__global__ __launch_bounds__(256) void mlp_loss_kernel(const float* Y, const float* T, const float* w,
                                                       int64_t M, float inv_norm, uint16_t* dY, double* loss) {
  __shared__ double red[4];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double l = 0.0;
  if (i < M) {
    const float wt = w ? w[i] : 1.f;
#pragma unroll
    for (int o = 0; o < MLP_OUT; ++o) {
      const float d = Y[i * MLP_OUTP + o] - T[i * MLP_OUT + o];
      dY[i * MLP_DYP + o] = f2bf(2.f * wt * d * inv_norm);
      l += (double)wt * d * d;
    }
#pragma unroll
    for (int o = MLP_OUT; o < MLP_DYP; ++o) dY[i * MLP_DYP + o] = 0;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(loss, (red[0] + red[1] + red[2] + red[3]) * (double)inv_norm);
}

__global__ void mlp_adam_kernel(float* p, const float* g, float* m, float* v, int n, float lr, float b1,
                                float b2, float eps, float bc1, float bc2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

// FP32 master -> BF16 operand copies (W1, W2, W3 and the transposes the
// backward pass reads), zero padding included.
__global__ void mlp_pack_kernel(const float* P, uint16_t* K) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= K_COUNT) return;
  float v = 0.f;
  if (i < K_W2) {
    const int r = (i - K_W1) / MLP_INP, c = (i - K_W1) % MLP_INP;
    v = c < MLP_IN ? P[P_W1 + r * MLP_IN + c] : 0.f;
  } else if (i < K_W3) {
    v = P[P_W2 + (i - K_W2)];
  } else if (i < K_W2T) {
    const int r = (i - K_W3) / MLP_H, c = (i - K_W3) % MLP_H;
    v = r < MLP_OUT ? P[P_W3 + r * MLP_H + c] : 0.f;
  } else if (i < K_W3T) {
    const int r = (i - K_W2T) / MLP_H, c = (i - K_W2T) % MLP_H;  // W2T[r][c] = W2[c][r]
    v = P[P_W2 + c * MLP_H + r];
  } else {
    const int r = (i - K_W3T) / MLP_DYP, c = (i - K_W3T) % MLP_DYP;  // W3T[r][c] = W3[c][r]
    v = c < MLP_OUT ? P[P_W3 + c * MLP_H + r] : 0.f;
  }
  K[i] = f2bf(v);
}

static inline unsigned nblk64(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }
// One workgroup (its LDS) per compute unit of an MI355X.
static inline unsigned row_workgroups(int64_t M) { return M < 256 * MLP_TILE ? nblk64(M, MLP_TILE) : 256u; }

void mlp_pack(hipStream_t st, const float* P, uint16_t* K) {
  hipLaunchKernelGGL(mlp_pack_kernel, dim3(nblk64(K_COUNT, 256)), dim3(256), 0, st, P, K);
}

void mlp_forward(hipStream_t st, const uint16_t* K, const float* P, const uint16_t* X, int64_t M, uint16_t* H1,
                 uint16_t* H2, float* Y) {
  if (M > 0)
    hipLaunchKernelGGL(mlp_forward_kernel, dim3(row_workgroups(M)), dim3(64 * ROW_WAVES), 0, st, K, P, X, M, H1, H2, Y);
}

// Splits of the weight gradients: at least 256 rows (two steps per wave),
// and at most 56: nine jobs each, two workgroups (their registers) on nearly
// every compute unit in one round (32,768 rows with 16 / 36 / 52 / 64 / 128
// splits: 53 / 34 / 28 / 32 / 40 us).  Without room for partial gradients they
// end in atomics, at most 16 splits of them.
int64_t mlp_wgrad_splits(int64_t M) {
  const int64_t s = (M + 255) / 256;
  return s < 56 ? s : 56;
}
size_t mlp_backward_workspace_bytes(int64_t M) { return sizeof(float) * P_COUNT * (size_t)mlp_wgrad_splits(M); }

void mlp_backward(hipStream_t st, const uint16_t* K, const uint16_t* X, int64_t M, const uint16_t* H1,
                  const uint16_t* H2, const uint16_t* dY, uint16_t* dH2, uint16_t* dH1, float* G, float* work) {
  if (M <= 0) return;
  hipLaunchKernelGGL(mlp_dgrad_kernel, dim3(row_workgroups(M)), dim3(64 * ROW_WAVES), 0, st, K, M, H1, H2, dY, dH2, dH1);
  int64_t splits = mlp_wgrad_splits(M);
  if (!work && splits > 16) splits = 16;
  const int64_t per = ((M + splits - 1) / splits + 127) / 128 * 128;
  splits = (M + per - 1) / per;
  WGradArgs g{M, per, X, H1, H2, dY, dH2, dH1, work ? work : G, work ? 0 : 1};
  hipLaunchKernelGGL(mlp_wgrad_kernel, dim3((unsigned)splits * WG_JOBS), dim3(256), 0, st, g);
  if (work)
    hipLaunchKernelGGL(mlp_reduce_kernel, dim3(nblk64(P_COUNT, 256)), dim3(256), 0, st, work, (int)splits, G);
}

void mlp_loss(hipStream_t st, const float* Y, const float* T, const float* w, int64_t M, float inv_norm,
              uint16_t* dY, double* loss) {
  if (M > 0) hipLaunchKernelGGL(mlp_loss_kernel, dim3(nblk64(M, 256)), dim3(256), 0, st, Y, T, w, M, inv_norm, dY, loss);
}

void mlp_adam(hipStream_t st, float* P, const float* G, float* m, float* v, int n, float lr, float b1, float b2,
              float eps, int step) {
  const float bc1 = 1.f - powf(b1, (float)step), bc2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(mlp_adam_kernel, dim3(nblk64(n, 256)), dim3(256), 0, st, P, G, m, v, n, lr, b1, b2, eps, bc1,
                     bc2);
}

}  // namespace mpm
