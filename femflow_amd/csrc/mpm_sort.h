// Host-side declarations of the binning primitives (mpm_sort.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "mpm355.h"

namespace mpm {

// How n keys of at most max_key are sorted: passes over digits of `bits` bits,
// and tiles of 256 * items keys, one workgroup each.
struct RadixPlan {
  int passes, bits, items;
  int64_t tiles;
};
RadixPlan radix_plan(int64_t n, uint32_t max_key);
size_t radix_workspace_bytes(int64_t n);  // for any key space
// Chunk list of a binning: occupied block b (bocc[b] != 0, particles
// bstart[b] .. bend[b]) gets chunks of at most `chunk` particles (a multiple
// of 256; start, count, b, block_scene[b]), numbered after those of the blocks
// before it; bfirst[b]
// and bcount[b] are its first chunk and chunk count (0 for empty blocks);
// nchunks[0] = the total.  plain: equal chunks (see FEW_ROWS).  part:
// chunk_list_part_words(nblocks) words.  split (may be null; plain only): the
// chunks once more, those of at most SMALL_CHUNK particles (nchunks[1] of them, 0
// if they are few) from the end of its split_cap entries, the others from the start.
constexpr int SMALL_CHUNK = 128, SPLIT_COUNT_BITS = 11;
size_t chunk_list_part_words(int64_t nblocks);
void chunk_list(const uint32_t* bocc, const uint32_t* bstart, const uint32_t* bend, const int* block_scene,
                int64_t nblocks, int chunk, uint32_t* part, int4* chunks, uint32_t* bfirst, uint32_t* bcount,
                uint32_t* nchunks, bool plain, int4* split, int64_t split_cap, hipStream_t st);
// The first pass's tile histogram inside the workspace, for a key kernel that
// also counts the first digit (rs_tile_histogram, mpm_sort_dev.h) and passes
// first_hist_done.
uint32_t* radix_first_hist(void* ws, int64_t n);
// Stable sort of source[0..n) carrying values: vals, or 0..n-1 when
// iota_values.  source is only read, and may be `keys`; keys and vals (n words
// each) are scratch.  The results (*kout, *vout) point into them or into the
// workspace; kout null: the sorted keys are not wanted.
void radix_sort(const RadixPlan& pl, const uint32_t* source, uint32_t* keys, uint32_t* vals, int64_t n, void* ws,
                bool iota_values, bool first_hist_done, uint32_t** kout, uint32_t** vout, hipStream_t st);
// Keys and the first pass's tile histogram (hist: radix_first_hist).
void bin_keys(const RadixPlan& pl, const float* x, int64_t n, int dim, int res, float inv_dx, int layout,
              uint32_t* keys, uint32_t* hist, hipStream_t st);

}  // namespace mpm
