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
// time and ended in a million device atomics (184 us).  Now: forward 29 us,
// dH 17 us, weight and bias gradients 38 + 6 us.
#include <hip/hip_runtime.h>

#include "mpm_mlp.h"

namespace mpm {

constexpr int MLP_TILE = 64;   // rows per workgroup of the row passes
constexpr int HSTR = MLP_H + 8;  // LDS row stride of an activation tile

// acc[u] (16 rows x 128 columns of one wave) += A B^T over K, A[row][k] from
// this lane's row pointer (global or LDS, already offset by lk), B row-major
// [128][ldb].  The next step's operands are in flight while this one's
// products run.
template <int K, typename PtrA>
__device__ __forceinline__ void mlp_layer(PtrA arow, const uint16_t* __restrict__ B, int ldb, int li, int lk,
                                          floatx4 (&acc)[8]) {
  const uint16_t* bp = B + (size_t)li * ldb + lk;
  uint4 a = *reinterpret_cast<const uint4*>(arow), b[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) b[u] = *reinterpret_cast<const uint4*>(bp + (size_t)16 * u * ldb);
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += 32) {
    uint4 an = a, bn[8];
    if (k0 + 32 < K) {
      an = *reinterpret_cast<const uint4*>(arow + k0 + 32);
#pragma unroll
      for (int u = 0; u < 8; ++u) bn[u] = *reinterpret_cast<const uint4*>(bp + (size_t)16 * u * ldb + k0 + 32);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] = mfma16x16x32(a, b[u], acc[u]);
    if (k0 + 32 < K) {
      a = an;
#pragma unroll
      for (int u = 0; u < 8; ++u) b[u] = bn[u];
    }
  }
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

// One wave: 16 rows through the three layers, hidden activations through LDS
// (and to memory for the backward pass).  The weights come from L2; what
// bounds it is the row load of X, 704 bytes per row.
__global__ __launch_bounds__(256) void mlp_forward_kernel(const uint16_t* __restrict__ K, const float* __restrict__ P,
                                                          const uint16_t* __restrict__ X, int64_t M,
                                                          uint16_t* __restrict__ H1, uint16_t* __restrict__ H2,
                                                          float* __restrict__ Y) {
  __shared__ __align__(16) uint16_t h_s[2][4][16 * HSTR];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int li = lane & 15, lk = (lane >> 4) * 8;
  const int64_t row0 = (int64_t)blockIdx.x * MLP_TILE + wv * 16;
  const int64_t arow = row0 + li < M ? row0 + li : M - 1;
  uint16_t *t1 = h_s[0][wv], *t2 = h_s[1][wv];
  floatx4 acc[8];
  zero_acc(acc);
  mlp_layer<MLP_INP>(X + arow * MLP_INP + lk, K + K_W1, MLP_INP, li, lk, acc);
  relu_tile(acc, P + P_B1, t1, lane);
  __syncthreads();
  zero_acc(acc);
  mlp_layer<MLP_H>(t1 + li * HSTR + lk, K + K_W2, MLP_H, li, lk, acc);
  tile_store(t1, H1, row0, M, lane);
  relu_tile(acc, P + P_B2, t2, lane);
  __syncthreads();
  tile_store(t2, H2, row0, M, lane);
  floatx4 y = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k0 = 0; k0 < MLP_H; k0 += 32)
    y = mfma16x16x32(*reinterpret_cast<const uint4*>(t2 + li * HSTR + k0 + lk),
                     *reinterpret_cast<const uint4*>(K + K_W3 + li * MLP_H + k0 + lk), y);
  if (li < MLP_OUT) {
    const float bb = P[P_B3 + li];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t row = row0 + (lane >> 4) * 4 + r;
      if (row < M) Y[row * MLP_OUTP + li] = y[r] + bb;
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

// dH2 = (dY W3) where H2 > 0, dH1 = (dH2 W2) where H1 > 0.
__global__ __launch_bounds__(256) void mlp_dgrad_kernel(const uint16_t* __restrict__ K, int64_t M,
                                                        const uint16_t* __restrict__ H1,
                                                        const uint16_t* __restrict__ H2,
                                                        const uint16_t* __restrict__ dY, uint16_t* __restrict__ dH2,
                                                        uint16_t* __restrict__ dH1) {
  __shared__ __align__(16) uint16_t h_s[2][4][16 * HSTR];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int li = lane & 15, lk = (lane >> 4) * 8;
  const int64_t row0 = (int64_t)blockIdx.x * MLP_TILE + wv * 16;
  const int64_t arow = row0 + li < M ? row0 + li : M - 1;
  uint16_t *t1 = h_s[0][wv], *t2 = h_s[1][wv];
  floatx4 acc[8];
  zero_acc(acc);
  mlp_layer<MLP_DYP>(dY + arow * MLP_DYP + lk, K + K_W3T, MLP_DYP, li, lk, acc);
  tile_load(t2, H2, row0, M, lane);
  tile_load(t1, H1, row0, M, lane);
  __syncthreads();
  mask_tile(acc, t2, lane);
  __syncthreads();
  zero_acc(acc);
  mlp_layer<MLP_H>(t2 + li * HSTR + lk, K + K_W2T, MLP_H, li, lk, acc);
  tile_store(t2, dH2, row0, M, lane);
  mask_tile(acc, t1, lane);
  __syncthreads();
  tile_store(t1, dH1, row0, M, lane);
}

// ------------------------------------------------------ weight gradients ----
// gW = dH^T In, a product over the rows.  Both operands are row-major with
// the rows as the reduction index, so a lane needs eight rows of one column
// per MFMA operand.  A lane loads 16 bytes (eight columns) of each of eight
// rows and transposes the 8 x 8 values in registers (one v_perm per pair),
// which gives the operands of eight tiles at once: tile t of lane li stands
// for column 8 li + t.  A wave then has a 128 x 128 block of the gradient in
// its accumulators, 64 products per 32 rows for 16 loads.
__device__ __forceinline__ void load_columns(const uint16_t* __restrict__ src, int64_t ld, int64_t k, int64_t kend,
                                             bool on, uint4 (&raw)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int64_t r = k + j < kend ? k + j : kend - 1;
    raw[j] = *reinterpret_cast<const uint4*>(src + r * ld);
    if (!on || k + j >= kend) raw[j] = make_uint4(0u, 0u, 0u, 0u);
  }
}
__device__ __forceinline__ void transpose8(const uint4 (&raw)[8], uint4 (&frag)[8]) {
  uint32_t f[8][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t lo[4] = {raw[2 * q].x, raw[2 * q].y, raw[2 * q].z, raw[2 * q].w};
    const uint32_t hi[4] = {raw[2 * q + 1].x, raw[2 * q + 1].y, raw[2 * q + 1].z, raw[2 * q + 1].w};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      f[2 * c][q] = __builtin_amdgcn_perm(hi[c], lo[c], 0x05040100u);
      f[2 * c + 1][q] = __builtin_amdgcn_perm(hi[c], lo[c], 0x07060302u);
    }
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) frag[t] = make_uint4(f[t][0], f[t][1], f[t][2], f[t][3]);
}

constexpr uint32_t BF_ONES = 0x3f803f80u;

struct WGradArgs {
  int64_t M, per;  // rows, rows per workgroup (a multiple of 128)
  const uint16_t *X, *H1, *H2, *dY, *dH2, *dH1;
  float* out;     // one gradient per split, or the gradient itself
  int atomic;     // add to `out` (one array) instead of storing a split's own
};

// Workgroup (split s, job): job 0..2 columns 128 job .. of gW1 (column 351,
// which holds no feature, is taken as 1 and gives the bias gradient), job 3
// gW2, job 4 gW3, gb3 and gb2.  Its four waves take a quarter of the split's
// rows each and add up through LDS.
__global__ __launch_bounds__(256, 1) void mlp_wgrad_kernel(WGradArgs g) {
  __shared__ __align__(16) floatx4 sum_s[2][64][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int li = lane & 15, grp = lane >> 4;
  const int job = blockIdx.y;
  const int64_t r0 = (int64_t)blockIdx.x * g.per, quarter = g.per / 4;
  const int64_t kb = r0 + wv * quarter;
  const int64_t ke = kb + quarter < g.M ? kb + quarter : g.M;
  float* const out = g.out + (g.atomic ? 0 : (int64_t)blockIdx.x * P_COUNT);
  auto put = [&](int i, float v) {
    if (g.atomic) atomicAdd(out + i, v);
    else out[i] = v;
  };
  if (job < 4) {
    const uint16_t* A = (job < 3 ? g.dH1 : g.dH2) + 8 * li;
    const uint16_t* B = job < 3 ? g.X : g.H1;
    const int64_t ldb = job < 3 ? MLP_INP : MLP_H;
    const int bc = (job < 3 ? 128 * job : 0) + 8 * li;
    const bool on = bc < ldb;
    B += on ? bc : 0;
    const bool ones = job == 2 && bc == MLP_IN - 7;  // this lane's tile 7 is column 351
    floatx4 acc[8][8];
#pragma unroll
    for (int ta = 0; ta < 8; ++ta) zero_acc(acc[ta]);
    uint4 ra[8], rb[8];
    if (kb < ke) {
      load_columns(A, MLP_H, kb + 8 * grp, ke, true, ra);
      load_columns(B, ldb, kb + 8 * grp, ke, on, rb);
    }
    for (int64_t k = kb; k < ke; k += 32) {
      uint4 fa[8], fb[8];
      transpose8(ra, fa);
      transpose8(rb, fb);
      if (ones) fb[7] = make_uint4(BF_ONES, BF_ONES, BF_ONES, BF_ONES);
      if (k + 32 < ke) {
        load_columns(A, MLP_H, k + 32 + 8 * grp, ke, true, ra);
        load_columns(B, ldb, k + 32 + 8 * grp, ke, on, rb);
      }
#pragma unroll
      for (int ta = 0; ta < 8; ++ta)
#pragma unroll
        for (int tb = 0; tb < 8; ++tb) acc[ta][tb] = mfma16x16x32(fa[ta], fb[tb], acc[ta][tb]);
    }
    // waves 2, 3 -> 0, 1; wave 1 -> 0
#pragma unroll
    for (int half = 2; half >= 1; half >>= 1) {
      if (wv >= half && wv < 2 * half) {
#pragma unroll
        for (int ta = 0; ta < 8; ++ta)
#pragma unroll
          for (int tb = 0; tb < 8; ++tb) sum_s[wv - half][ta * 8 + tb][lane] = acc[ta][tb];
      }
      __syncthreads();
      if (wv < half) {
#pragma unroll
        for (int ta = 0; ta < 8; ++ta)
#pragma unroll
          for (int tb = 0; tb < 8; ++tb) acc[ta][tb] += sum_s[wv][ta * 8 + tb][lane];
      }
      __syncthreads();
    }
    float* nat = reinterpret_cast<float*>(sum_s);  // [128][129]
    if (wv == 0) {
#pragma unroll
      for (int ta = 0; ta < 8; ++ta)
#pragma unroll
        for (int tb = 0; tb < 8; ++tb)
#pragma unroll
          for (int r = 0; r < 4; ++r) nat[(8 * (grp * 4 + r) + ta) * 129 + 8 * li + tb] = acc[ta][tb][r];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 128 * 128; e += 256) {
      const int m = e >> 7, n = e & 127;
      const float v = nat[m * 129 + n];
      if (job == 3) put(P_W2 + m * MLP_H + n, v);
      else if (128 * job + n < MLP_IN) put(P_W1 + m * MLP_IN + 128 * job + n, v);
      else if (128 * job + n == MLP_IN) put(P_B1 + m, v);
    }
    return;
  }
  // job 4: A = dY (three columns) with B = H2 and 1; A = dH2 with B = 1
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

// G += the sum of the splits' gradients, in split order.
__global__ __launch_bounds__(256) void mlp_reduce_kernel(const float* __restrict__ part, int splits,
                                                         float* __restrict__ G) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P_COUNT) return;
  float s = 0.f;
#pragma unroll 16
  for (int k = 0; k < splits; ++k) s += part[(int64_t)k * P_COUNT + i];
  G[i] += s;
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

void mlp_pack(hipStream_t st, const float* P, uint16_t* K) {
  hipLaunchKernelGGL(mlp_pack_kernel, dim3(nblk64(K_COUNT, 256)), dim3(256), 0, st, P, K);
}

void mlp_forward(hipStream_t st, const uint16_t* K, const float* P, const uint16_t* X, int64_t M, uint16_t* H1,
                 uint16_t* H2, float* Y) {
  if (M > 0)
    hipLaunchKernelGGL(mlp_forward_kernel, dim3(nblk64(M, MLP_TILE)), dim3(256), 0, st, K, P, X, M, H1, H2, Y);
}

// Splits of the weight gradients: at least 256 rows (two steps per wave),
// and at most 64 (with five jobs each, 320 workgroups: a little over one per
// CU; more would only add partial gradients to write and read).  Without
// room for partial gradients they end in atomics, at most 16 splits of them.
int64_t mlp_wgrad_splits(int64_t M) {
  const int64_t s = (M + 255) / 256;
  return s < 64 ? s : 64;
}
size_t mlp_backward_workspace_bytes(int64_t M) { return sizeof(float) * P_COUNT * (size_t)mlp_wgrad_splits(M); }

void mlp_backward(hipStream_t st, const uint16_t* K, const uint16_t* X, int64_t M, const uint16_t* H1,
                  const uint16_t* H2, const uint16_t* dY, uint16_t* dH2, uint16_t* dH1, float* G, float* work) {
  if (M <= 0) return;
  hipLaunchKernelGGL(mlp_dgrad_kernel, dim3(nblk64(M, MLP_TILE)), dim3(256), 0, st, K, M, H1, H2, dY, dH2, dH1);
  int64_t splits = mlp_wgrad_splits(M);
  if (!work && splits > 16) splits = 16;
  const int64_t per = ((M + splits - 1) / splits + 127) / 128 * 128;
  splits = (M + per - 1) / per;
  WGradArgs g{M, per, X, H1, H2, dY, dH2, dH1, work ? work : G, work ? 0 : 1};
  hipLaunchKernelGGL(mlp_wgrad_kernel, dim3((unsigned)splits, 5), dim3(256), 0, st, g);
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
