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
// works through a chunk in rows of CHUNK_ROW particles, one per thread, so a
// block's particles are cut into R = ceil(count / CHUNK_ROW) rows of nearly
// equal size first (chunks of 333 would take two rows each for the work of
// 1.3).  Either every row is a chunk, or the rows of a block are grouped into
// chunks of up to `chunk` particles: a row by itself finishes sooner and
// leaves a shorter tail; a pair loads and stages one arena for both and
// spreads a wave's lanes over twice as many cells, which is what counts where
// a cell holds dozens of particles (the lanes that share one add to the same
// words).  One choice for the whole list: chunks of one and of two rows side
// by side were the slowest (2^20 particles 5,464 us, see below).  Two launches
// over tiles of SCAN_THREADS blocks, one block per thread (coalesced reads,
// a few hundred tiles for a 128^3 grid): per-tile counts, then each tile adds
// the counts of the tiles before it, scans its own blocks and writes their
// chunks, first chunk and chunk count.
constexpr uint32_t CHUNK_ROW = 256;
// Rows are grouped where most of them are in blocks of more than 18 particles
// per cell.  48 substeps, all rows single / grouped, in us: 100,003 particles
// at 17 per cell 1,500 / 1,723; 400,000 at 17 2,839 / 2,978; 524,288 at 10
// 3,425 / 3,908; 262,144 at 21 2,210 / 2,118; 2^20 at 21 5,581 / 5,164;
// 131,072 at 62 1,744 / 1,638.
constexpr uint32_t GROUP_ABOVE = 18 * 64;
// And single up to this many rows in all, one and a half per compute unit of
// an MI355X: fewer, larger chunks would leave units without one (16,384
// particles at 8 per cell 1,035 / 1,230).
// Engines of many scenes (plain) cut a block into ceil(count / chunk) equal
// chunks, without regard to rows: their tens of thousands of chunks come from
// contended ticket queues, and single rows cost more there (64 scenes, 24
// substeps with upload and download: 16,112 single, 14,827 rows grouped,
// 15,160 plain; grouping moves the fixed-point scale of scenes with a fraction
// of a particle per cell, whose light nodes it then decides).  Engines with
// the corrector are plain too: its features and activations round to BF16, so
// another fixed-point scale now and then moves a light node's velocity gradient
// by 1e-3 (262,144 particles in 5,400 cells: no difference in time).
constexpr uint32_t FEW_ROWS = 384;
// Small chunks go to the launch of their own (split) from this many on, one round
// of four-wave workgroups (three per compute unit): fewer find room beside the
// others, and a second pass over the few takes longer than they do there.  Us per
// substep of engines at 16 particles per cell, all apart / none: 8 scenes of
// 16,384 (231 small of 619 chunks) 46 / 36, 16 of 32,768 (16 of 1,483) 76 / 61; at
// 1 per cell, all chunks small, 8 scenes of 4,096 (959) 29 / 37, 8 of 32,768 (5,743)
// 69 / 107.  (Before there was a second launch: 43, 69, 55, 124.)
constexpr uint32_t APART_FROM = 768;

// Of a block (or their sums over a tile): rows, chunks with rows grouped, rows
// in dense blocks.  A block's pairs that would be less than 3/4 full stay
// single (260 particles: 130 + 130, not 256 + 4).
struct BlockRows {
  uint32_t rows, chunks, dense, small;
};
__device__ __forceinline__ BlockRows block_rows(const uint32_t* __restrict__ bocc, const uint32_t* __restrict__ bstart,
                                                const uint32_t* __restrict__ bend, int64_t b, uint32_t per_chunk,
                                                int plain) {
  if (!bocc[b]) return {0u, 0u, 0u, 0u};
  const uint32_t cnt = bend[b] - bstart[b], rows = (cnt + CHUNK_ROW - 1u) / CHUNK_ROW;
  if (plain) {
    const uint32_t c = (cnt + per_chunk * CHUNK_ROW - 1u) / (per_chunk * CHUNK_ROW);
    return {c, c, 0u, cnt <= (uint32_t)SMALL_CHUNK ? 1u : 0u};  // (a small block is one chunk)
  }
  const bool group = 4u * cnt >= 3u * CHUNK_ROW * rows;
  return {rows, group ? (rows + per_chunk - 1u) / per_chunk : rows, cnt > GROUP_ABOVE ? rows : 0u, 0u};
}

__global__ __launch_bounds__(SCAN_THREADS) void block_tile_kernel(const uint32_t* __restrict__ bocc,
                                                                  const uint32_t* __restrict__ bstart,
                                                                  const uint32_t* __restrict__ bend,
                                                                  int64_t nblocks, uint32_t per_chunk,
                                                                  uint4* __restrict__ part, int plain) {
  __shared__ uint32_t sh[SCAN_THREADS];
  const int64_t b = (int64_t)blockIdx.x * SCAN_THREADS + threadIdx.x;
  const BlockRows r = b < nblocks ? block_rows(bocc, bstart, bend, b, per_chunk, plain) : BlockRows{0u, 0u, 0u, 0u};
  uint32_t rows, chunks, dense, small;
  block_exclusive_scan(r.rows, sh, &rows);
  block_exclusive_scan(r.chunks, sh, &chunks);
  block_exclusive_scan(r.dense, sh, &dense);
  block_exclusive_scan(r.small, sh, &small);
  if (threadIdx.x == 0) part[blockIdx.x] = make_uint4(rows, chunks, dense, small);
}

__global__ __launch_bounds__(SCAN_THREADS) void block_chunks_kernel(
    const uint32_t* __restrict__ bocc, const uint32_t* __restrict__ bstart, const uint32_t* __restrict__ bend,
    const int* __restrict__ block_scene, int64_t nblocks, uint32_t per_chunk, const uint4* __restrict__ part,
    int4* __restrict__ chunks, uint32_t* __restrict__ bfirst, uint32_t* __restrict__ bcount,
    uint32_t* __restrict__ nchunks, int plain, int4* __restrict__ split, uint32_t split_cap) {
  __shared__ uint32_t sh[SCAN_THREADS];
  uint32_t rows_before = 0, chunks_before = 0, small_before = 0, rows = 0, dense = 0, small = 0;
  for (uint32_t q = threadIdx.x; q < gridDim.x; q += SCAN_THREADS) {
    const uint4 v = part[q];
    rows += v.x;
    dense += v.z;
    small += v.w;
    if (q < blockIdx.x) {
      rows_before += v.x;
      chunks_before += v.y;
      small_before += v.w;
    }
  }
  uint32_t rows_all, dense_all, before;
  block_exclusive_scan(rows, sh, &rows_all);
  block_exclusive_scan(dense, sh, &dense_all);
  // the same in every workgroup
  const bool single = !plain && (rows_all <= FEW_ROWS || 2u * dense_all < rows_all);
  block_exclusive_scan(single ? rows_before : chunks_before, sh, &before);
  const int64_t b = (int64_t)blockIdx.x * SCAN_THREADS + threadIdx.x;
  BlockRows r = b < nblocks ? block_rows(bocc, bstart, bend, b, per_chunk, plain) : BlockRows{0u, 0u, 0u, 0u};
  const uint32_t c = single ? r.rows : r.chunks;
  uint32_t tot;
  const uint32_t run = block_exclusive_scan(c, sh, &tot) + before;
  uint32_t small_run = 0;
  if (split) {
    uint32_t small_all, first;
    block_exclusive_scan(small, sh, &small_all);
    if (small_all < APART_FROM) r.small = small_before = 0u;
    block_exclusive_scan(small_before, sh, &first);
    small_run = block_exclusive_scan(r.small, sh, &tot) + first;
  }
  if (b < nblocks) {
    bfirst[b] = run;
    bcount[b] = c;
    if (c) {
      const uint32_t p0 = bstart[b], cnt = bend[b] - p0;
      const int sc = block_scene[b];
      uint32_t s0 = 0, s1;
      for (uint32_t j = 0; j < c; ++j, s0 = s1) {
        // its rows end at r1 (64 bits: rows^2 leaves 32 from 2^24 particles in one block on)
        const uint32_t r1 = (uint32_t)((uint64_t)r.rows * (j + 1u) / c);
        s1 = (uint32_t)((uint64_t)cnt * r1 / r.rows);
        chunks[run + j] = make_int4((int)(p0 + s0), (int)(s1 - s0), (int)b, sc);
        if (split)
          split[r.small ? split_cap - 1u - small_run : run + j - small_run] =
              make_int4((int)(p0 + s0), (int)((s1 - s0) | ((uint32_t)sc << SPLIT_COUNT_BITS)), (int)b, (int)(run + j));
      }
    }
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == SCAN_THREADS - 1) {
    nchunks[0] = run + c;
    nchunks[1] = small_run + r.small;
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

size_t chunk_list_part_words(int64_t nblocks) { return 4 * ((size_t)cdiv(nblocks, SCAN_THREADS) + 1); }

void chunk_list(const uint32_t* bocc, const uint32_t* bstart, const uint32_t* bend, const int* block_scene,
                int64_t nblocks, int chunk, uint32_t* part, int4* chunks, uint32_t* bfirst, uint32_t* bcount,
                uint32_t* nchunks, bool plain, int4* split, int64_t split_cap, hipStream_t st) {
  if (nblocks <= 0) return;
  const unsigned tiles = (unsigned)cdiv(nblocks, SCAN_THREADS);
  const uint32_t per_chunk = (uint32_t)chunk / CHUNK_ROW;
  uint4* part4 = reinterpret_cast<uint4*>(part);
  hipLaunchKernelGGL(block_tile_kernel, dim3(tiles), dim3(SCAN_THREADS), 0, st, bocc, bstart, bend, nblocks,
                     per_chunk, part4, plain ? 1 : 0);
  hipLaunchKernelGGL(block_chunks_kernel, dim3(tiles), dim3(SCAN_THREADS), 0, st, bocc, bstart, bend,
                     block_scene, nblocks, per_chunk, part4, chunks, bfirst, bcount, nchunks, plain ? 1 : 0, split, (uint32_t)split_cap);
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
