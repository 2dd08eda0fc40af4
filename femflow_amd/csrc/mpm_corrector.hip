// Learned grid corrector inside the engine's substep.
//
// With the corrector on, every substep (taken at dt_big) runs
//   transfer (G2P(n-1) + P2G(n)) -> cellf_kernel -> grid update (also
//   writing each node's P2G momentum/mass) -> corrector_kernel
// and corrector_kernel, for each active block, gathers the
// 3x3x3-node stencil features of the block's 64 nodes into LDS, runs the
// 351 -> 128 -> 128 -> 3 MLP on MFMA (BF16 operands, FP32 accumulate) and
// adds the predicted correction, scaled down on nodes with little mass, to
// the nodes' updated velocities (re-clamped, walls re-applied), then clears
// the block's cell sums for the next substep.
// In sampling mode corrector_sample_kernel writes the features (and the updated
// velocity) of every node with mass instead: the training data.
//
// Features of node n, for each neighbour o = (d0, d1, d2) in {-1, 0, 1}^3 in
// lexicographic order, 13 values: m / m_ref, p / (m_ref v_ref) (3), and the
// mass-weighted mean deformation gradient of the particles whose stencil base
// is node n + o, minus I (9; zero when that cell is empty).  Output: the
// velocity correction divided by v_ref.
#include <hip/hip_runtime.h>

#include "mpm_engine.h"
#include "mpm_engine_kernels.h"
#include "mpm_math.h"
#include "mpm_mlp.h"

namespace mpm {

struct CorrArgs {
  const uint16_t* packed;  // BF16 operands (corr_pack_kernel)
  const float* params;     // FP32 master (biases read from here)
  float inv_mref, inv_pref, vref;
  CorrExtract ex;          // ex.X != null: sampling mode
  uint32_t* count;
};

// ------------------------------------------------------------ cell sums ----
// Particles in binned order: the lanes of a wave mostly share cells, so the
// wave sums runs of equal cells (segmented scan over lanes) and only the
// last lane of each run adds to global memory.
__global__ __launch_bounds__(256) void cellf_kernel(EngineArgs a, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  uint32_t key = 0xffffffffu;
  float val[10];
#pragma unroll
  for (int c = 0; c < 10; ++c) val[c] = 0.f;
  if (i < n) {
    const SceneDev sc = a.scenes[a.s.attr[i] >> 8];
    float x[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) x[d] = a.s.x[tix(i, 3, d)];
    int base[3];
    float fx[3];
    if (locate3(x, sc, base, fx)) {
      key = (uint32_t)node_addr(sc, base[0], base[1], base[2]);
      const float m = a.s.mass[i];
      val[0] = m;
#pragma unroll
      for (int e = 0; e < 9; ++e) val[1 + e] = m * a.s.F[tix(i, 9, e)];
    }
  }
  const uint32_t prev = __shfl_up(key, 1);
  const bool head = lane == 0 || prev != key;
  const uint64_t heads = __ballot(head);
  const int seg = __popcll(heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1ull)));
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int sup = __shfl_up(seg, off);
#pragma unroll
    for (int c = 0; c < 10; ++c) {
      const float up = __shfl_up(val[c], off);
      if (lane >= off && sup == seg) val[c] += up;
    }
  }
  const int snext = __shfl_down(seg, 1);
  const bool tail = lane == 63 || snext != seg;
  if (tail && key != 0xffffffffu) {
    float* dst = reinterpret_cast<float*>(a.cellf + (size_t)key * 3);
#pragma unroll
    for (int c = 0; c < 10; ++c) atomicAdd(dst + c, val[c]);
    mark_active(a, key >> 6);
  }
}

// ----------------------------------------------------------- corrector ----
// The correction applied to a node is scaled by min(1, m / (CORR_GATE m_ref)):
// nodes with little mass (surfaces) keep the plain big step's velocity.
constexpr float CORR_GATE = 0.25f;
constexpr int HS = 136;  // LDS row stride of the hidden tile (BF16)
constexpr int XS = 360;  // and of the feature tile

// The weights in the order of the MFMA operands, 16 bytes per lane: element
// ((step * N / 16 + u) * 64 + lane) * 8 + j is W[16 u + lane % 16][k], k =
// 32 step + 8 (lane / 16) + j.
constexpr int CORR_STEPS = MLP_INP / 32;
constexpr int CK_W1 = 0, CK_W2 = CK_W1 + CORR_STEPS * 32 * MLP_H, CK_W3 = CK_W2 + MLP_H * MLP_H,
              CK_COUNT = CK_W3 + MLP_OUTP * MLP_H;

__global__ void corr_pack_kernel(const float* P, uint16_t* K) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= CK_COUNT) return;
  const int base = i < CK_W2 ? CK_W1 : (i < CK_W3 ? CK_W2 : CK_W3), tiles = i < CK_W3 ? MLP_H / 16 : 1;
  const int e = i - base, j = e & 7, lane = (e >> 3) & 63, tile = e >> 9;
  const int col = 16 * (tile % tiles) + (lane & 15), k = 32 * (tile / tiles) + 8 * (lane >> 4) + j;
  float v = 0.f;
  if (i < CK_W2) {
    if (k < MLP_IN) v = P[P_W1 + col * MLP_IN + k];
  } else if (i < CK_W3) {
    v = P[P_W2 + col * MLP_H + k];
  } else if (col < MLP_OUT) {
    v = P[P_W3 + col * MLP_H + k];
  }
  K[i] = f2bf(v);
}

struct BlockAt {
  SceneDev sc;
  int bi, bj, bk;
};
__device__ __forceinline__ BlockAt block_at(const EngineArgs& a, uint32_t g) {
  BlockAt at;
  at.sc = a.scenes[a.nscenes == 1 ? 0 : a.block_scene[g]];
  const int local = (int)g - at.sc.block_base, nb = at.sc.nb;
  at.bi = local / (nb * nb);
  at.bj = (local / nb) % nb;
  at.bk = local % nb;
  return at;
}

// Raw values of node t of the 6x6x6 neighbourhood of a block (t < 216)
struct NodeRaw {
  float4 q, c0, c1, c2;
};
__device__ __forceinline__ NodeRaw node_raw(const EngineArgs& a, const BlockAt& at, int t) {
  NodeRaw n;
  n.q = n.c0 = n.c1 = n.c2 = make_float4(0.f, 0.f, 0.f, 0.f);
  const int gi = at.bi * 4 - 1 + t / 36, gj = at.bj * 4 - 1 + (t / 6) % 6, gk = at.bk * 4 - 1 + t % 6;
  const int res = at.sc.res;
  if (t < 216 && gi >= 0 && gj >= 0 && gk >= 0 && gi <= res && gj <= res && gk <= res) {
    const size_t na = node_addr(at.sc, gi, gj, gk);
    n.q = a.pm[na];  // zero outside this substep's active blocks
    n.c0 = a.cellf[na * 3];
    n.c1 = a.cellf[na * 3 + 1];
    n.c2 = a.cellf[na * 3 + 2];
  }
  return n;
}

// Its 13 normalised features
__device__ __forceinline__ void write_record(const NodeRaw& n, const CorrArgs& c, uint16_t* rec) {
  float f[13];
#pragma unroll
  for (int e = 0; e < 13; ++e) f[e] = 0.f;
  if (n.q.w > 0.f) {
    f[0] = n.q.w * c.inv_mref;
    f[1] = n.q.x * c.inv_pref;
    f[2] = n.q.y * c.inv_pref;
    f[3] = n.q.z * c.inv_pref;
  }
  if (n.c0.x > 0.f) {
    const float im = 1.f / n.c0.x;
    const float F[9] = {n.c0.y, n.c0.z, n.c0.w, n.c1.x, n.c1.y, n.c1.z, n.c1.w, n.c2.x, n.c2.y};
#pragma unroll
    for (int e = 0; e < 9; ++e) f[4 + e] = F[e] * im - ((e % 4 == 0) ? 1.f : 0.f);
  }
#pragma unroll
  for (int e = 0; e < 13; ++e) rec[e] = f2bf(f[e]);
}

// Feature f of block node r: its place among the neighbourhood's records (for
// the padding feature the 14th value of the last one, which is zero).
__device__ __forceinline__ uint32_t feature_at(int r, int f) {
  if (f >= MLP_IN) return 216 * 13;
  const int o = f / 13, first = (r >> 4) * 36 + ((r >> 2) & 3) * 6 + (r & 3);
  return (uint32_t)((first + (o / 9) * 36 + ((o / 3) % 3) * 6 + o % 3) * 13 + f % 13);
}

// One workgroup per compute unit, eight waves, over the active blocks; wave
// (rg, ch) holds 16 of the block's 64 nodes and 64 of the 128 columns.  W1
// stays in LDS (88 KB), W2, W3, the biases and the places of a thread's share
// of the features in registers for the whole launch, and the next block's
// neighbourhood is in flight while this one's layers run.  Blocks none of
// whose nodes have mass (a third of the candidates of three cubes on an 80^3
// grid) end after the records.  What bounds it: the barriers and LDS round
// trips of about four blocks in turn.  262,144 particles, 80^3: 74 us with the
// weights read from L2 without prefetch and every block taken, 30 now.
// The products are summed in the features' own order.  (Records padded to 16
// values, from which layer 1 can take its operands without the feature tile,
// take 24 us, but their other order of sums rounds now and then to another
// BF16 activation, which moves a light node's velocity gradient by 1e-3.)
constexpr int CORR_THREADS = 512;
struct CorrShared {
  uint4 w1[CORR_STEPS * 8 * 64];
  uint16_t x[64 * XS];
  uint16_t rec[216 * 13 + 8];
  uint16_t h[64 * HS];
  uint32_t live[2][4];  // by turn and wave: a node of the block has mass
};
__global__ __launch_bounds__(CORR_THREADS) void corrector_kernel(EngineArgs a, CorrArgs c) {
  __shared__ __align__(16) CorrShared sh;
  const int t = threadIdx.x;
  const int lane = t & 63, wv = t >> 6, rg = wv & 3, ch = wv >> 2;
  const int li = lane & 15, lk = (lane >> 4) * 8;
  const uint32_t ncand = *a.cand_count;
  const uint32_t count = ncand + *a.list_count;
  if (blockIdx.x >= count) return;
  const uint4* const packed = reinterpret_cast<const uint4*>(c.packed);
#pragma unroll
  for (int e = 0; e < CORR_STEPS * 8 * 64 / CORR_THREADS; ++e)
    sh.w1[e * CORR_THREADS + t] = packed[CK_W1 / 8 + e * CORR_THREADS + t];
  uint4 w2[MLP_H / 32][4], w3[MLP_H / 32];
  float b1[4], b2[4];
#pragma unroll
  for (int k = 0; k < MLP_H / 32; ++k) {
#pragma unroll
    for (int u = 0; u < 4; ++u) w2[k][u] = packed[CK_W2 / 8 + (k * 8 + 4 * ch + u) * 64 + lane];
    w3[k] = packed[CK_W3 / 8 + k * 64 + lane];
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    b1[u] = c.params[P_B1 + 64 * ch + 16 * u + li];
    b2[u] = c.params[P_B2 + 64 * ch + 16 * u + li];
  }
  const float b3 = c.params[P_B3 + (li < MLP_OUT ? li : 0)];
  // this thread's node of the neighbourhood, and whether it is the block's own
  const int n0 = t / 36, n1 = (t / 6) % 6, n2 = t % 6;
  const bool own = t < 216 && n0 >= 1 && n0 <= 4 && n1 >= 1 && n1 <= 4 && n2 >= 1 && n2 <= 4;
  // the pairs of features that this thread copies into the tile
  constexpr int PAIRS = 64 * (MLP_INP / 2) / CORR_THREADS;
  static_assert(PAIRS * CORR_THREADS == 64 * (MLP_INP / 2), "whole rounds");
  uint32_t from[PAIRS];  // two places of 16 bits
#pragma unroll
  for (int j = 0; j < PAIRS; ++j) {
    const int e = j * CORR_THREADS + t, r = e / (MLP_INP / 2), f = 2 * (e % (MLP_INP / 2));
    from[j] = feature_at(r, f) | (feature_at(r, f + 1) << 16);
  }
  if (t == 0) sh.rec[216 * 13] = 0;
  const uint16_t *const xrow = sh.x + (16 * rg + li) * XS + lk, *const hrow = sh.h + (16 * rg + li) * HS + lk;
  uint32_t b = blockIdx.x, g = active_block(a, b, ncand);
  BlockAt at = block_at(a, g);
  NodeRaw raw = node_raw(a, at, t);
  for (int turn = 0;; turn ^= 1) {
    if (t < 216) write_record(raw, c, sh.rec + 13 * t);
    const bool live = __ballot(own && raw.q.w > 0.f) != 0ull;
    if (wv < 4 && lane == 0) sh.live[turn][wv] = live ? 1u : 0u;
    // (the records of the turn before were read up to the barrier ahead of its
    // layer 1, its flags up to this one)
    __syncthreads();
    const uint32_t any = (sh.live[turn][0] | sh.live[turn][1]) | (sh.live[turn][2] | sh.live[turn][3]);
    const BlockAt here = at;
    const uint32_t ghere = g;
    b += gridDim.x;
    const bool more = b < count;
    if (more) {
      g = active_block(a, b, ncand);
      at = block_at(a, g);
      raw = node_raw(a, at, t);
    }
    if (any) {
#pragma unroll
      for (int j = 0; j < PAIRS; ++j) {
        const int e = j * CORR_THREADS + t, r = e / (MLP_INP / 2), f = 2 * (e % (MLP_INP / 2));
        *reinterpret_cast<uint32_t*>(sh.x + r * XS + f) =
            (uint32_t)sh.rec[from[j] & 0xffffu] | ((uint32_t)sh.rec[from[j] >> 16] << 16);
      }
      // the nodes that this lane corrects, for the end
      float mn[4], vel[4];
      const bool writes = ch == 0 && li < MLP_OUT;
      float4* const own_vel = a.vel + (size_t)ghere * 64 + 16 * rg + (lane >> 4) * 4;
      if (writes) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          mn[r] = a.pm[(size_t)ghere * 64 + 16 * rg + (lane >> 4) * 4 + r].w;
          vel[r] = reinterpret_cast<const float*>(own_vel + r)[li];
        }
      }
      auto relu_rows = [&](const floatx4(&acc)[4], const float(&bias)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = acc[u][r] + bias[u];
            sh.h[(16 * rg + (lane >> 4) * 4 + r) * HS + 64 * ch + 16 * u + li] = f2bf(v > 0.f ? v : 0.f);
          }
      };
      __syncthreads();
      floatx4 acc[4];
      // layer 1: 352 -> 128 (ReLU)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < CORR_STEPS; ++k) {
        const uint4 av = *reinterpret_cast<const uint4*>(xrow + 32 * k);
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[u] = mfma16x16x32(av, sh.w1[(k * 8 + 4 * ch + u) * 64 + lane], acc[u]);
      }
      relu_rows(acc, b1);
      __syncthreads();
      // layer 2: 128 -> 128 (ReLU)
      uint4 hv[MLP_H / 32];
#pragma unroll
      for (int k = 0; k < MLP_H / 32; ++k) hv[k] = *reinterpret_cast<const uint4*>(hrow + 32 * k);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < MLP_H / 32; ++k)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[u] = mfma16x16x32(hv[k], w2[k][u], acc[u]);
      __syncthreads();
      relu_rows(acc, b2);
      __syncthreads();
      // layer 3: 128 -> 3, add to the node velocities
      if (ch == 0) {
        floatx4 y = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < MLP_H / 32; ++k) y = mfma16x16x32(*reinterpret_cast<const uint4*>(hrow + 32 * k), w3[k], y);
        if (writes) {
          const SceneDev& sc = here.sc;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (!(mn[r] > 0.f)) continue;
            const int nr = 16 * rg + (lane >> 4) * 4 + r;
            const int I[3] = {here.bi * 4 + (nr >> 4), here.bj * 4 + ((nr >> 2) & 3), here.bk * 4 + (nr & 3)};
            const float gate = tmin(1.f, mn[r] * c.inv_mref * (1.f / CORR_GATE));
            float v = vel[r] + gate * (y[r] + b3) * c.vref;
            v = tmin(tmax(v, -sc.v_allowed), sc.v_allowed);
            if (sc.boundary == MPM_BC_REFERENCE) {
              if (I[li] < 1 || I[li] >= sc.res - 1) v = 0.f;
            } else {
#pragma unroll
              for (int d = 0; d < 3; ++d)
                if (I[d] < sc.bound || I[d] > sc.res - sc.bound) v = 0.f;
            }
            if (I[0] > sc.res || I[1] > sc.res || I[2] > sc.res) v = 0.f;
            reinterpret_cast<float*>(own_vel + r)[li] = v;
          }
        }
      }
    }
    if (!more) return;
  }
}

// Sampling: every node with mass becomes one training row of features (and
// its velocity), in the network's own order.
__global__ __launch_bounds__(256) void corrector_sample_kernel(EngineArgs a, CorrArgs c) {
  __shared__ uint16_t rec_s[216 * 13 + 8];
  __shared__ uint32_t row_s[64];
  const int t = threadIdx.x;
  const uint32_t ncand = *a.cand_count;
  const uint32_t count = ncand + *a.list_count;
  for (uint32_t b = blockIdx.x; b < count; b += gridDim.x) {
    const uint32_t g = active_block(a, b, ncand);
    const BlockAt at = block_at(a, g);
    if (t < 216) write_record(node_raw(a, at, t), c, rec_s + 13 * t);
    if (t == 0) rec_s[216 * 13] = 0;
    if (t < 64) {
      const size_t na = (size_t)g * 64 + t;
      uint32_t row = 0xffffffffu;
      if (a.pm[na].w > 0.f) {
        row = atomicAdd(c.count, 1u);
        if ((int64_t)row < c.ex.max_rows) {
          const float4 v = a.vel[na];
          c.ex.nodes[row] = (uint32_t)na;
          c.ex.vel[3 * (size_t)row] = v.x;
          c.ex.vel[3 * (size_t)row + 1] = v.y;
          c.ex.vel[3 * (size_t)row + 2] = v.z;
        } else {
          row = 0xffffffffu;
        }
      }
      row_s[t] = row;
    }
    __syncthreads();
    for (int idx = t; idx < 64 * (MLP_INP / 2); idx += 256) {
      const int r = idx / (MLP_INP / 2), f = 2 * (idx % (MLP_INP / 2));
      const uint32_t row = row_s[r];
      if (row == 0xffffffffu) continue;
      reinterpret_cast<uint32_t*>(c.ex.X + (size_t)row * MLP_INP)[f / 2] =
          (uint32_t)rec_s[feature_at(r, f)] | ((uint32_t)rec_s[feature_at(r, f + 1)] << 16);
    }
    __syncthreads();
  }
}

// Clear the cell sums and P2G records of this substep's active blocks
// (every cell that received a particle lies in one: cellf_kernel marks it),
// so that blocks outside the next substep's active set read as empty.
__global__ __launch_bounds__(256) void cellf_clear_kernel(EngineArgs a) {
  const uint32_t ncand = *a.cand_count;
  const uint32_t count = ncand + *a.list_count;
  const int t = threadIdx.x;
  for (uint32_t b = blockIdx.x; b < count; b += gridDim.x) {
    const uint32_t g = active_block(a, b, ncand);
    float4* p = a.cellf + (size_t)g * 64 * 3;
    if (t < 192) p[t] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (t < 64) a.pm[(size_t)g * 64 + t] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

__global__ void gather_vel_kernel(const float4* vel, const uint32_t* nodes, int64_t count, float* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const float4 v = vel[nodes[i]];
  out[3 * i] = v.x;
  out[3 * i + 1] = v.y;
  out[3 * i + 2] = v.z;
}

static inline unsigned cblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

void Engine::launch_cellf(hipStream_t s, const EngineArgs& a) {
  if (n > 0) hipLaunchKernelGGL(cellf_kernel, dim3(cblk(n, 256)), dim3(256), 0, s, a, n);
}

void Engine::launch_corrector(hipStream_t s, const EngineArgs& a, const CorrExtract* ex) {
  CorrArgs c{};
  c.packed = d_corr_packed;
  c.params = d_corr_params;
  c.inv_mref = 1.f / corr_mref;
  c.inv_pref = 1.f / (corr_mref * corr_vref);
  c.vref = corr_vref;
  if (ex) c.ex = *ex;
  c.count = d_corr_count;
  if (ex) hipLaunchKernelGGL(corrector_sample_kernel, dim3(num_cus * 2), dim3(256), 0, s, a, c);
  else hipLaunchKernelGGL(corrector_kernel, dim3(num_cus), dim3(CORR_THREADS), 0, s, a, c);
  hipLaunchKernelGGL(cellf_clear_kernel, dim3(num_cus * 2), dim3(256), 0, s, a);
}

int Engine::set_corrector(const float* params, float m_ref, float v_ref, int enable) {
  if ((enable && !params) || (params && (!(m_ref > 0.f) || !(v_ref > 0.f)))) {
    set_error("mpm_ctx_set_corrector: needs parameters and positive m_ref, v_ref");
    return MPM_ERR_ARG;
  }
  hipStreamSynchronize(own_stream);
  drop_graphs();
  int rc;
  if ((enable || params) && !d_pm) {
    const size_t nodes = (size_t)total_blocks * 64;
    if ((rc = alloc((void**)&d_pm, sizeof(float4) * nodes))) return rc;
    if ((rc = alloc((void**)&d_cellf, sizeof(float4) * 3 * nodes))) return rc;
    if ((rc = alloc((void**)&d_corr_params, sizeof(float) * P_COUNT))) return rc;
    if ((rc = alloc((void**)&d_corr_packed, sizeof(uint16_t) * CK_COUNT))) return rc;
    if ((rc = alloc((void**)&d_corr_count, sizeof(uint32_t) * 4))) return rc;
    // zero on the engine's own (non-blocking) stream, before any of its work
    fill_u32(own_stream, reinterpret_cast<uint32_t*>(d_cellf), (int64_t)nodes * 12, 0u);
    fill_u32(own_stream, reinterpret_cast<uint32_t*>(d_pm), (int64_t)nodes * 4, 0u);
    if (hipStreamSynchronize(own_stream) != hipSuccess) {
      set_error("mpm_ctx_set_corrector: clearing the feature buffers failed");
      return MPM_ERR_HIP;
    }
  }
  corr_on = enable != 0;
  if (params) {
    corr_mref = m_ref;
    corr_vref = v_ref;
    // the caller's parameters are ready on its stream: order the copy after
    // it, on the engine's stream (a device-to-device hipMemcpy would run on
    // the null stream, unordered with the engine's non-blocking stream)
    if (hipEventRecord(ev_in, user_stream) != hipSuccess || hipStreamWaitEvent(own_stream, ev_in, 0) != hipSuccess ||
        hipMemcpyAsync(d_corr_params, params, sizeof(float) * P_COUNT, hipMemcpyDeviceToDevice, own_stream) !=
            hipSuccess) {
      set_error("mpm_ctx_set_corrector: parameter copy failed");
      return MPM_ERR_HIP;
    }
    hipLaunchKernelGGL(corr_pack_kernel, dim3(cblk(CK_COUNT, 256)), dim3(256), 0, own_stream, d_corr_params, d_corr_packed);
    if (hipStreamSynchronize(own_stream) != hipSuccess) {
      set_error("mpm_ctx_set_corrector: pack failed");
      return MPM_ERR_HIP;
    }
  }
  return MPM_OK;
}

// One P2G + grid update from the current state (particles unchanged), then
// the corrector's features of every node with mass.  X == null: stop after
// the grid update, applying the corrector if it is enabled
// (grid_velocity() then reads node velocities).
int Engine::corrector_sample(uint16_t* X, uint32_t* nodes, float* vel, int64_t max_rows, int64_t* rows) {
  if (!d_pm) {
    set_error("mpm_corrector_sample: set a corrector (mpm_ctx_set_corrector) first");
    return MPM_ERR_ARG;
  }
  const bool was_on = corr_on;
  corr_on = true;
  hipStream_t s = own_stream;
  if (hipEventRecord(ev_in, user_stream) != hipSuccess || hipStreamWaitEvent(s, ev_in, 0) != hipSuccess) {
    corr_on = was_on;
    set_error("mpm_corrector_sample: stream setup failed");
    return MPM_ERR_HIP;
  }
  enqueue_bin(s, 1, 0, true);  // also starts the one-substep segment
  since_bin = 0;  // freshly binned: the next run continues from this order
  chunks_plain = true;
  const EngineArgs a = args(nullptr, 0, 0);
  {
    EngineArgs a0 = a;
    a0.perm = pending_perm;  // this P2G moves the particles into binned order
    a0.rec = in_records ? d_rec : nullptr;
    in_records = false;
    pending_perm = nullptr;
    launch_transfer(0, s, a0);
  }
  launch_cellf(s, a);
  launch_grid(s, a, 0, 1, 0);
  fill_u32(s, d_corr_count, 1, 0u);
  CorrExtract ex{X, nodes, vel, max_rows};
  if (X) {
    launch_corrector(s, a, &ex);  // features only
  } else if (was_on) {
    launch_corrector(s, a, nullptr);  // the substep's corrected grid velocity
  } else {
    hipLaunchKernelGGL(cellf_clear_kernel, dim3(num_cus * 2), dim3(256), 0, s, a);
  }
  corr_on = was_on;
  uint32_t cnt = 0;
  if (hipMemcpyAsync(&cnt, d_corr_count, sizeof(uint32_t), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess) {
    set_error("mpm_corrector_sample: kernel failure");
    return MPM_ERR_HIP;
  }
  if (rows) *rows = (int64_t)cnt;
  return MPM_OK;
}

int Engine::grid_velocity(const uint32_t* nodes, int64_t count, float* out) {
  if (count <= 0) return MPM_OK;
  hipLaunchKernelGGL(gather_vel_kernel, dim3(cblk(count, 256)), dim3(256), 0, own_stream, d_vel, nodes, count, out);
  if (hipStreamSynchronize(own_stream) != hipSuccess) {
    set_error("mpm_grid_velocity: kernel failure");
    return MPM_ERR_HIP;
  }
  return MPM_OK;
}

}  // namespace mpm
