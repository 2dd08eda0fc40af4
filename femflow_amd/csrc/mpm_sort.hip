// Cell binning: key generation, a stable LSD radix sort on 32-bit keys
// (digits of 8 to 11 bits; three launches per pass: tile histograms, a per-digit scan
// over tiles, the stable scatter), and the chunk list (a two-launch scan of
// per-block chunk counts) that gives the engine its work items for the
// transfer kernels.
//
// Stability: inside a tile each wave owns a contiguous run of keys and walks
// it in index order; ranks among equal digits come from a 64-lane match mask
// built with one ballot per digit bit plus per-wave running counters, and
// waves are ordered by a prefix over their counters.  Tiles are ordered by
// the per-digit exclusive scan over tiles of the per-tile histograms.  Each
// pass is therefore a stable counting sort, and the whole sort equals a
// stable sort by key.
#include "mpm_sort.h"
#include "mpm_sort_dev.h"

namespace mpm {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

// Per-tile digit histogram, written tile-major: hist[(tile << bits) + d].
template <int ITEMS>
__global__ __launch_bounds__(RS_THREADS) void rs_upsweep(const uint32_t* __restrict__ keys,
                                                         int64_t n, int shift, int bits,
                                                         uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[RS_MAX_BINS];
  const int64_t base = (int64_t)blockIdx.x * (ITEMS * RS_THREADS);
  // every key of the thread in flight at once: one memory round trip per
  // tile rather than one per few rounds
  uint32_t k[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t idx = base + (int64_t)r * RS_THREADS + threadIdx.x;
    k[r] = keys[idx < n ? idx : 0];
  }
  rs_tile_histogram<ITEMS>(k, n, shift, bits, h, hist);
}

// Exclusive prefix sum over the 256 threads of a workgroup (one value each):
// wave-level inclusive scans by lane shuffles, then the wave totals.
__device__ __forceinline__ uint32_t excl_scan_256(uint32_t v, uint32_t* wave_tot) {
  const int t = threadIdx.x;
  const int lane = t & 63, w = t >> 6;
  uint32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(incl, (unsigned)off);
    if (lane >= off) incl += y;
  }
  if (lane == 63) wave_tot[w] = incl;
  __syncthreads();
  uint32_t base = 0;
#pragma unroll
  for (int i = 0; i < RS_WAVES; ++i) base += i < w ? wave_tot[i] : 0u;
  return base + incl - v;
}

// Per digit d: the exclusive prefix over tiles of the tile-major histogram
// hist[tile * bins + d] (written to offs in the same layout) and the
// digit's total (dtot[d]); the scatter adds the exclusive prefix of the
// totals over digits.  A workgroup takes DS_DIGITS digits (neighbouring lanes,
// so that every read and write is whole 64-byte pieces of rows) and splits the
// tiles into DS_GROUPS contiguous ranges: each group sums its range, the sums
// are prefixed in LDS, and each group then writes its range's running prefix.
// The serial walk is what bounds it, so the ranges are many and short: 512
// tiles of 2,048 digits in groups of 8 tiles on 128 workgroups; with 64 digits
// and 16 ranges per workgroup (32 of 32 tiles) it took 9.3 us.
constexpr int DS_DIGITS = 16, DS_GROUPS = 64;
__global__ __launch_bounds__(DS_DIGITS * DS_GROUPS) void rs_digit_scan(const uint32_t* __restrict__ hist, int ntiles,
                                                                       int bits, uint32_t* __restrict__ offs,
                                                                       uint32_t* __restrict__ dtot) {
  __shared__ uint32_t part[DS_GROUPS][DS_DIGITS];
  const int dl = threadIdx.x % DS_DIGITS, g = threadIdx.x / DS_DIGITS;
  const int d = blockIdx.x * DS_DIGITS + dl;
  const int per = (ntiles + DS_GROUPS - 1) / DS_GROUPS;
  const int t0 = g * per < ntiles ? g * per : ntiles;
  const int t1 = t0 + per < ntiles ? t0 + per : ntiles;
  uint32_t sum = 0;
#pragma unroll 8
  for (int tl = t0; tl < t1; ++tl) sum += hist[((int64_t)tl << bits) + d];
  part[g][dl] = sum;
  __syncthreads();
  uint32_t run = 0;
  const int used = ntiles < DS_GROUPS ? ntiles : DS_GROUPS;
#pragma unroll 8
  for (int i = 0; i < used; ++i) run += i < g ? part[i][dl] : 0u;
  if (g == DS_GROUPS - 1) dtot[d] = run + sum;
#pragma unroll 8
  for (int tl = t0; tl < t1; ++tl) {
    const uint32_t v = hist[((int64_t)tl << bits) + d];
    offs[((int64_t)tl << bits) + d] = run;
    run += v;
  }
}

// Tile of a workgroup: each XCD (workgroup id mod 8) takes a contiguous run of
// tiles, whose keys of one digit are neighbours in the output, so that their
// partial lines meet in that XCD's L2.
__device__ __forceinline__ uint32_t xcd_tile() {
  const uint32_t xcd = blockIdx.x & 7u, per = gridDim.x >> 3, rem = gridDim.x & 7u;
  return xcd * per + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
}

// kout null: the sorted keys are not wanted.
template <int ITEMS>
__global__ __launch_bounds__(RS_THREADS) void rs_downsweep(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin, uint32_t* __restrict__ kout,
    uint32_t* __restrict__ vout, int64_t n, int shift, int bits, const uint32_t* __restrict__ offs,
    const uint32_t* __restrict__ dtot, int iota_values) {
  __shared__ uint32_t cnt[RS_WAVES][RS_MAX_BINS];
  __shared__ uint32_t goff[RS_MAX_BINS];
  __shared__ uint32_t wt[RS_WAVES];
  const int t = threadIdx.x;
  const int w = t >> 6;
  const unsigned lane = __lane_id();
  constexpr int MAX_DPT = RS_MAX_BINS / RS_THREADS;
  const int bins = 1 << bits, dpt = bins / RS_THREADS;  // digits per thread
  // keys and values of the wave's run in flight from the start
  const uint32_t tile = xcd_tile();
  const int64_t base = (int64_t)tile * (ITEMS * RS_THREADS) + (int64_t)w * 64 * ITEMS;
  uint32_t k[ITEMS], val[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t idx = base + r * 64 + lane, at = idx < n ? idx : 0;
    k[r] = kin[at];
    val[r] = iota_values ? (uint32_t)idx : vin[at];
  }
#pragma unroll
  for (int i = 0; i < RS_WAVES; ++i)
    for (int d = t; d < bins; d += RS_THREADS) cnt[i][d] = 0;
  // global start of digit d in this tile: keys of smaller digits (all tiles)
  // plus keys of digit d in earlier tiles; thread t takes digits
  // t * dpt .. t * dpt + dpt - 1
  {
    uint32_t tot[MAX_DPT], before[MAX_DPT], sum = 0;
#pragma unroll
    for (int j = 0; j < MAX_DPT; ++j) {
      if (j >= dpt) break;
      tot[j] = dtot[t * dpt + j];
      before[j] = offs[((int64_t)tile << bits) + t * dpt + j];
      sum += tot[j];
    }
    uint32_t run = excl_scan_256(sum, wt);
#pragma unroll
    for (int j = 0; j < MAX_DPT; ++j) {
      if (j >= dpt) break;
      goff[t * dpt + j] = run + before[j];
      run += tot[j];
    }
  }
  __syncthreads();
  uint32_t rank[ITEMS];
  const uint64_t lt = lanemask_lt();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t idx = base + r * 64 + lane;
    const bool valid = idx < n;
    const uint32_t d = (k[r] >> shift) & (uint32_t)(bins - 1);
    const uint64_t vm = __ballot(valid);
    const uint64_t m = match_digit(d, bits, vm);
    uint32_t prev = 0;
    if (valid) prev = cnt[w][d];
    rank[r] = prev + (uint32_t)__popcll(m & lt);
    if (valid && lane == 63u - (unsigned)__clzll(m)) cnt[w][d] = prev + (uint32_t)__popcll(m);
  }
  __syncthreads();
  for (int d = t; d < bins; d += RS_THREADS) {
    uint32_t run = 0;
#pragma unroll
    for (int i = 0; i < RS_WAVES; ++i) {
      const uint32_t c = cnt[i][d];
      cnt[i][d] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t idx = base + r * 64 + lane;
    if (idx < n) {
      const uint32_t d = (k[r] >> shift) & (uint32_t)(bins - 1);
      const uint32_t dst = goff[d] + cnt[w][d] + rank[r];
      if (kout) kout[dst] = k[r];
      vout[dst] = val[r];
    }
  }
}

// ---------------------------------------------------------------- scan ----
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* sh, uint32_t* total) {
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int off = 1; off < SCAN_THREADS; off <<= 1) {
    const uint32_t a = t >= off ? sh[t - off] : 0u;
    __syncthreads();
    sh[t] += a;
    __syncthreads();
  }
  const uint32_t incl = sh[t];
  *total = sh[SCAN_THREADS - 1];
  __syncthreads();
  return incl - v;
}

// ------------------------------------------------------- chunk list ----
// Chunk list of the new binning, numbered over blocks.  A transfer workgroup
// works through a chunk in steps of CHUNK_ROW particles, one per thread, and
// loads, clears and stages an arena for it: a chunk costs about 1.4 steps beside
// its own.  Three ways to cut a block, one for the whole list:
// - plain: ceil(count / chunk) equal chunks, the fewest (but 333 particles take
//   two steps for the work of 1.3);
// - single: rows of nearly equal size, ceil(count / CHUNK_ROW) of them, each a
//   chunk: the fewest steps and the shortest tail, at most twice the chunks;
// - grouped: those rows in chunks of up to `chunk` particles; pairs that would be
//   less than 3/4 full stay single (260 particles: 130 + 130, not 256 + 4).
// Two launches over tiles of SCAN_THREADS blocks, one block per thread
// (coalesced reads, a few hundred tiles for a 128^3 grid): per-tile sums, then
// each tile adds those of the tiles before it, scans its own blocks and writes
// their chunks, first chunk and chunk count.
constexpr uint32_t CHUNK_ROW = 256;
// A block is dense above this (18 particles per cell).
constexpr uint32_t GROUP_ABOVE = 18 * 64;
// The rule, for engines of one scene without the corrector.  R rows in all, T steps
// of the plain list, 768 chunks running at once on an MI355X (three per compute
// unit); us per substep, plain / single / grouped, one elastic body:
// - R <= 384: single; fewer, larger chunks would leave units without one.  20,000
//   particles at 8 per cell 21.2 / 17.6 / 21.1.
// - most rows in dense blocks: grouped up to R = 2,100 (200,000 at 64 per cell 34.9 /
//   38.4 / 30.5, at 20 30.2 / 30.8 / 29.3), where its fewer steps leave a shorter
//   tail; beyond, plain (2^20 in three bodies at 20 75.0 / 83.5 / 79.4, 1,600,000 at
//   32 95.7 / 114.7 / 99.9, at 64 93.5 / 115.7 / 91.6).
// - else up to one round of chunks, R <= 768, single (100,000 at 12 25.5 / 21.2 / 24.9),
//   and up to 2,100 where it saves a tenth of the steps, 10 T >= 11 R (300,000 in
//   three bodies at 18, T = 1.16 R, 39.2 / 34.9 / 37.4; but 200,000 at 14, 1.04 R, 27.0
//   / 29.9 / 29.7); beyond, plain: the chunks' arenas are what counts (800,000 at 6
//   and 16 66.0 / 80.4 / 75.9, 60.0 / 65.4 / 60.2; 4,000,000 at 8 291 / 335 / 323).
// Engines of many scenes are plain: their tens of thousands of chunks come from
// contended ticket queues, and single rows cost more there (64 scenes, 24
// substeps with upload and download: 16,112 single, 14,827 rows grouped,
// 15,160 plain; grouping moves the fixed-point scale of scenes with a fraction
// of a particle per cell, whose light nodes it then decides).  Engines with
// the corrector are plain too: its features and activations round to BF16, so
// another fixed-point scale now and then moves a light node's velocity gradient
// by 1e-3 (262,144 particles in 5,400 cells: no difference in time).
constexpr uint32_t FEW_ROWS = 384, ONE_ROUND = 768, FEW_ROUNDS = 2100;
// Small chunks go to the launch of their own (split) from this many on, one round
// of four-wave workgroups (three per compute unit): fewer find room beside the
// others, and a second pass over the few takes longer than they do there.  Us per
// substep of engines at 16 particles per cell, all apart / none: 8 scenes of
// 16,384 (231 small of 619 chunks) 46 / 36, 16 of 32,768 (16 of 1,483) 76 / 61; at
// 1 per cell, all chunks small, 8 scenes of 4,096 (959) 29 / 37, 8 of 32,768 (5,743)
// 69 / 107.  (Before there was a second launch: 43, 69, 55, 124.)
constexpr uint32_t APART_FROM = 768;

// Of a block, or their sums: rows, chunks with rows grouped, plain chunks, plain
// chunks of at most SMALL_CHUNK, steps of the plain chunks, rows in dense blocks.
enum { CUT_ROWS, CUT_GROUPED, CUT_PLAIN, CUT_SMALL, CUT_STEPS, CUT_DENSE, CUTS };
typedef uint32_t BlockCuts[CUTS];
__device__ __forceinline__ void block_cuts(const uint32_t* __restrict__ bocc, const uint32_t* __restrict__ bstart,
                                           const uint32_t* __restrict__ bend, int64_t b, int64_t nblocks,
                                           uint32_t per_chunk, BlockCuts& r) {
#pragma unroll
  for (int i = 0; i < CUTS; ++i) r[i] = 0u;
  if (b >= nblocks || !bocc[b]) return;
  const uint32_t cnt = bend[b] - bstart[b], rows = (cnt + CHUNK_ROW - 1u) / CHUNK_ROW;
  const uint32_t plain = (rows + per_chunk - 1u) / per_chunk;
  const bool group = 4ull * cnt >= 3ull * CHUNK_ROW * rows;
  r[CUT_ROWS] = rows;
  r[CUT_GROUPED] = group ? plain : rows;
  r[CUT_PLAIN] = plain;
  r[CUT_SMALL] = cnt <= (uint32_t)SMALL_CHUNK ? 1u : 0u;  // (a small block is one chunk)
  r[CUT_STEPS] = plain * (((cnt + plain - 1u) / plain + CHUNK_ROW - 1u) / CHUNK_ROW);
  r[CUT_DENSE] = cnt > GROUP_ABOVE ? rows : 0u;
}

// Sums over the 256 threads of a workgroup, to every thread.
template <int K>
__device__ __forceinline__ void block_sums(uint32_t (&v)[K], uint32_t (*sh)[K]) {
#pragma unroll
  for (int i = 0; i < K; ++i) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v[i] += __shfl_xor(v[i], o);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][i] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < K; ++i) v[i] = (sh[0][i] + sh[1][i]) + (sh[2][i] + sh[3][i]);
}

constexpr int PART_WORDS = 8;  // per tile: its BlockCuts

__global__ __launch_bounds__(SCAN_THREADS) void block_tile_kernel(const uint32_t* __restrict__ bocc,
                                                                  const uint32_t* __restrict__ bstart,
                                                                  const uint32_t* __restrict__ bend,
                                                                  int64_t nblocks, uint32_t per_chunk,
                                                                  uint32_t* __restrict__ part) {
  __shared__ uint32_t sh[SCAN_THREADS / 64][CUTS];
  BlockCuts r;
  block_cuts(bocc, bstart, bend, (int64_t)blockIdx.x * SCAN_THREADS + threadIdx.x, nblocks, per_chunk, r);
  block_sums<CUTS>(r, sh);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < CUTS; ++i) part[(size_t)blockIdx.x * PART_WORDS + i] = r[i];
  }
}

__global__ __launch_bounds__(SCAN_THREADS) void block_chunks_kernel(
    const uint32_t* __restrict__ bocc, const uint32_t* __restrict__ bstart, const uint32_t* __restrict__ bend,
    const int* __restrict__ block_scene, int64_t nblocks, uint32_t per_chunk, const uint32_t* __restrict__ part,
    int4* __restrict__ chunks, uint32_t* __restrict__ bfirst, uint32_t* __restrict__ bcount,
    uint32_t* __restrict__ nchunks, int plain, int4* __restrict__ split, uint32_t split_cap) {
  __shared__ uint32_t sh[SCAN_THREADS], sums_s[SCAN_THREADS / 64][2 * CUTS];
  uint32_t sums[2 * CUTS];  // over all tiles, over those before this one
#pragma unroll
  for (int i = 0; i < 2 * CUTS; ++i) sums[i] = 0u;
  for (uint32_t q = threadIdx.x; q < gridDim.x; q += SCAN_THREADS) {
    const uint4 lo = reinterpret_cast<const uint4*>(part)[2 * q], hi = reinterpret_cast<const uint4*>(part)[2 * q + 1];
    const BlockCuts v = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y};
#pragma unroll
    for (int i = 0; i < CUTS; ++i) {
      sums[i] += v[i];
      sums[CUTS + i] += q < blockIdx.x ? v[i] : 0u;
    }
  }
  block_sums<2 * CUTS>(sums, sums_s);
  const int64_t b = (int64_t)blockIdx.x * SCAN_THREADS + threadIdx.x;
  BlockCuts r;
  block_cuts(bocc, bstart, bend, b, nblocks, per_chunk, r);
  // the cut (the same in every workgroup)
  const uint32_t R = sums[CUT_ROWS];
  const bool dense = 2u * sums[CUT_DENSE] >= R, few = R <= FEW_ROUNDS;
  const bool single = !plain && (R <= FEW_ROWS || (!dense && (R <= ONE_ROUND || (few && 10ull * sums[CUT_STEPS] >= 11ull * R))));
  const bool grouped = !plain && !single && dense && few;
  const int cut = single ? CUT_ROWS : (grouped ? CUT_GROUPED : CUT_PLAIN);
  const uint32_t c = single ? r[CUT_ROWS] : (grouped ? r[CUT_GROUPED] : r[CUT_PLAIN]);
  const uint32_t before = cut == CUT_ROWS ? sums[CUTS + CUT_ROWS]
                                          : (cut == CUT_GROUPED ? sums[CUTS + CUT_GROUPED] : sums[CUTS + CUT_PLAIN]);
  const uint32_t pieces = single || grouped ? r[CUT_ROWS] : r[CUT_PLAIN];  // equal parts that chunks are made of
  uint32_t tot;
  const uint32_t run = block_exclusive_scan(c, sh, &tot) + before;
  uint32_t small = 0, small_run = 0;
  if (split) {  // (plain)
    const bool apart = sums[CUT_SMALL] >= APART_FROM;
    small = apart ? r[CUT_SMALL] : 0u;
    small_run = block_exclusive_scan(small, sh, &tot) + (apart ? sums[CUTS + CUT_SMALL] : 0u);
  }
  if (b < nblocks) {
    bfirst[b] = run;
    bcount[b] = c;
    if (c) {
      const uint32_t p0 = bstart[b], cnt = bend[b] - p0;
      const int sc = block_scene[b];
      uint32_t s0 = 0, s1;
      for (uint32_t j = 0; j < c; ++j, s0 = s1) {
        // its pieces end at r1 (64 bits: rows^2 leaves 32 from 2^24 particles in one block on)
        const uint32_t r1 = (uint32_t)((uint64_t)pieces * (j + 1u) / c);
        s1 = (uint32_t)((uint64_t)cnt * r1 / pieces);
        chunks[run + j] = make_int4((int)(p0 + s0), (int)(s1 - s0), (int)b, sc);
        if (split)
          split[small ? split_cap - 1u - small_run : run + j - small_run] =
              make_int4((int)(p0 + s0), (int)((s1 - s0) | ((uint32_t)sc << SPLIT_COUNT_BITS)), (int)b, (int)(run + j));
      }
    }
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == SCAN_THREADS - 1) {
    nchunks[0] = run + c;
    nchunks[1] = small_run + small;
  }
}

// ---------------------------------------------------------------- keys ----
// base = trunc(fl32(fl32(x*inv_dx) - 0.5)), clamped to [0, res] (the same
// rounding the reference's (x*inv_dx - 0.5).astype(int64) sees on FP32 x).
__device__ __forceinline__ int cell_coord(float x, float inv_dx, int res) {
  const float s = __fmul_rn(x, inv_dx);
  const float t = __fsub_rn(s, 0.5f);
  int b;
  if (!(t > -1.0f)) b = 0;            // also NaN
  else if (!(t < (float)res)) b = res;
  else b = (int)t;                    // truncation toward zero
  return b < 0 ? 0 : (b > res ? res : b);
}

template <int DIM>
__device__ __forceinline__ uint32_t bin_key(const float* x, int res, float inv_dx, int layout) {
  int b[DIM];
#pragma unroll
  for (int d = 0; d < DIM; ++d) b[d] = cell_coord(x[d], inv_dx, res);
  const uint32_t r1 = (uint32_t)res + 1u;
  uint32_t key;
  if (layout == MPM_KEY_ROWMAJOR) {
    key = (uint32_t)b[0];
#pragma unroll
    for (int d = 1; d < DIM; ++d) key = key * r1 + (uint32_t)b[d];
  } else {
    const uint32_t nb = (r1 + 3u) / 4u;
    uint32_t bid = (uint32_t)(b[0] >> 2), cid = (uint32_t)(b[0] & 3);
#pragma unroll
    for (int d = 1; d < DIM; ++d) {
      bid = bid * nb + (uint32_t)(b[d] >> 2);
      cid = cid * 4u + (uint32_t)(b[d] & 3);
    }
    key = bid * (DIM == 3 ? 64u : 16u) + cid;
  }
  return key;
}

// Keys of one sort tile per workgroup, with the tile's histogram of the first
// digit (the sort then starts at its scan: one launch and one read of the keys
// fewer).
template <int DIM, int ITEMS>
__global__ __launch_bounds__(RS_THREADS) void bin_keys_kernel(const float* __restrict__ x, int64_t n, int res,
                                                              float inv_dx, int layout, uint32_t* __restrict__ keys,
                                                              int bits, uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[RS_MAX_BINS];
  const int64_t base = (int64_t)blockIdx.x * (ITEMS * RS_THREADS);
  float px[ITEMS][DIM];
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
    k[r] = bin_key<DIM>(px[r], res, inv_dx, layout);
    if (i < n) keys[i] = k[r];
  }
  rs_tile_histogram<ITEMS>(k, n, 0, bits, h, hist);
}

// ------------------------------------------------------------ host side ----
static inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Keys per thread: the fewest that keep the tiles within MAX_SMALL_TILES, since
// a tile's rounds of ranking are a serial chain and few tiles leave most of the
// chip idle; the histograms (one row of digits per tile) bound it from above.
// mpm_bin at 4 / 8 / 16 keys in us: 4,096 keys 28 / 36 / 54; 131,072 32 / 39 /
// 57; 524,288 56 / 57 / 72; 2^20 86 / 72 / 82; 2^21 142 / 113 / 103.
constexpr int64_t MAX_SMALL_TILES = 512;
static int radix_items(int64_t n) {
  if (n <= MAX_SMALL_TILES * RS_THREADS * 4) return 4;
  return n <= MAX_SMALL_TILES * RS_THREADS * 8 ? 8 : 16;
}

RadixPlan radix_plan(int64_t n, uint32_t max_key) {
  int bits = 0;
  while (bits < 32 && (max_key >> bits) != 0u) ++bits;
  RadixPlan p;
  p.passes = bits == 0 ? 1 : (bits + RS_MAX_BITS - 1) / RS_MAX_BITS;
  p.bits = (bits + p.passes - 1) / p.passes;
  if (p.bits < 8) p.bits = 8;  // one digit per thread of the scatter's offsets
  p.items = radix_items(n);
  p.tiles = cdiv(n > 0 ? n : 1, (int64_t)RS_THREADS * p.items);
  return p;
}

// Words of one tile histogram table, enough for any key space and for any
// count up to n (a caller may sort fewer keys in the same workspace).
static size_t radix_hist_words(int64_t n) {
  const int64_t small = cdiv(n > 0 ? n : 1, RS_THREADS * 4), large = cdiv(n > 0 ? n : 1, RS_THREADS * 16);
  const int64_t most = small < MAX_SMALL_TILES ? small : MAX_SMALL_TILES;
  return (size_t)RS_MAX_BINS * (size_t)(large > most ? large : most);
}

size_t radix_workspace_bytes(int64_t n) {
  // keys and values (ping-pong) + histogram + its prefix + digit totals
  return sizeof(uint32_t) * (2 * (size_t)(n > 0 ? n : 0) + 2 * radix_hist_words(n) + RS_MAX_BINS);
}

size_t chunk_list_part_words(int64_t nblocks) { return PART_WORDS * ((size_t)cdiv(nblocks, SCAN_THREADS) + 1); }

void chunk_list(const uint32_t* bocc, const uint32_t* bstart, const uint32_t* bend, const int* block_scene,
                int64_t nblocks, int chunk, uint32_t* part, int4* chunks, uint32_t* bfirst, uint32_t* bcount,
                uint32_t* nchunks, bool plain, int4* split, int64_t split_cap, hipStream_t st) {
  if (nblocks <= 0) return;
  const unsigned tiles = (unsigned)cdiv(nblocks, SCAN_THREADS);
  const uint32_t per_chunk = (uint32_t)chunk / CHUNK_ROW;
  hipLaunchKernelGGL(block_tile_kernel, dim3(tiles), dim3(SCAN_THREADS), 0, st, bocc, bstart, bend, nblocks,
                     per_chunk, part);
  hipLaunchKernelGGL(block_chunks_kernel, dim3(tiles), dim3(SCAN_THREADS), 0, st, bocc, bstart, bend,
                     block_scene, nblocks, per_chunk, part, chunks, bfirst, bcount, nchunks, plain ? 1 : 0, split,
                     (uint32_t)split_cap);
}

uint32_t* radix_first_hist(void* ws, int64_t n) { return (uint32_t*)ws + 2 * n; }

template <int ITEMS>
static void radix_pass(const RadixPlan& pl, int pass, bool hist_done, const uint32_t* kin, const uint32_t* vin,
                       uint32_t* kout, uint32_t* vout, int64_t n, uint32_t* hist, uint32_t* offs, uint32_t* dtot,
                       bool iota, hipStream_t st) {
  const int shift = pl.bits * pass;
  const dim3 tiles((unsigned)pl.tiles);
  if (!hist_done)
    hipLaunchKernelGGL((rs_upsweep<ITEMS>), tiles, dim3(RS_THREADS), 0, st, kin, n, shift, pl.bits, hist);
  hipLaunchKernelGGL(rs_digit_scan, dim3((1u << pl.bits) / DS_DIGITS), dim3(DS_DIGITS * DS_GROUPS), 0, st, hist, (int)pl.tiles,
                     pl.bits, offs, dtot);
  hipLaunchKernelGGL((rs_downsweep<ITEMS>), tiles, dim3(RS_THREADS), 0, st, kin, vin, kout, vout, n, shift, pl.bits,
                     offs, dtot, iota ? 1 : 0);
}

void radix_sort(const RadixPlan& pl, const uint32_t* source, uint32_t* keys, uint32_t* vals, int64_t n, void* ws,
                bool iota_values, bool first_hist_done, uint32_t** kout, uint32_t** vout, hipStream_t st) {
  uint32_t* hist = radix_first_hist(ws, n);
  uint32_t* offs = hist + radix_hist_words(n);
  uint32_t* dtot = offs + radix_hist_words(n);
  const uint32_t *ka = source, *va = vals;
  uint32_t *kb = (uint32_t*)ws, *vb = (uint32_t*)ws + n, *knext = keys, *vnext = vals;
  for (int p = 0; p < pl.passes; ++p) {
    uint32_t* ko = !kout && p == pl.passes - 1 ? nullptr : kb;
    const bool done = p == 0 && first_hist_done, iota = iota_values && p == 0;
    if (pl.items == 4) radix_pass<4>(pl, p, done, ka, va, ko, vb, n, hist, offs, dtot, iota, st);
    else if (pl.items == 8) radix_pass<8>(pl, p, done, ka, va, ko, vb, n, hist, offs, dtot, iota, st);
    else radix_pass<16>(pl, p, done, ka, va, ko, vb, n, hist, offs, dtot, iota, st);
    ka = kb;
    va = vb;
    uint32_t* t;
    t = kb; kb = knext; knext = t;
    t = vb; vb = vnext; vnext = t;
  }
  // the last pass's outputs
  if (kout) *kout = knext;
  *vout = vnext;
}

void bin_keys(const RadixPlan& pl, const float* x, int64_t n, int dim, int res, float inv_dx, int layout,
              uint32_t* keys, uint32_t* hist, hipStream_t st) {
  if (n <= 0) return;
#define MPM_BIN_KEYS(D, I)                                                                                      \
  hipLaunchKernelGGL((bin_keys_kernel<D, I>), dim3((unsigned)pl.tiles), dim3(RS_THREADS), 0, st, x, n, res,     \
                     inv_dx, layout, keys, pl.bits, hist)
  if (dim == 3) {
    if (pl.items == 4) MPM_BIN_KEYS(3, 4);
    else if (pl.items == 8) MPM_BIN_KEYS(3, 8);
    else MPM_BIN_KEYS(3, 16);
  } else {
    if (pl.items == 4) MPM_BIN_KEYS(2, 4);
    else if (pl.items == 8) MPM_BIN_KEYS(2, 8);
    else MPM_BIN_KEYS(2, 16);
  }
#undef MPM_BIN_KEYS
}

}  // namespace mpm
