// sort.h — LDS-ranked LSD radix sort of (u64 key, u32 value) pairs and a
// device exclusive scan, used for Morton codes, the active contact list and
// the per-vertex contact incidence.
#pragma once

#include "common.h"

namespace cloth {

struct SortScratch {
  uint32_t* hist = nullptr;  // radix_hist_entries of the largest sort
  size_t hist_cap = 0;
  bool block_sort = false;   // sort_setup found the LDS for sorts in one work-group
};

// Whether this device has the LDS for k_sort_block (and prepares it).
bool sort_setup();

// Stable sort of n pairs on key bits [begin_bit, end_bit).  Sorts in place
// between (keys, vals) and (keys_tmp, vals_tmp); returns true when the result
// ended up in the *_tmp buffers.
bool radix_sort_pairs(hipStream_t st, uint64_t* keys, uint32_t* vals, uint64_t* keys_tmp, uint32_t* vals_tmp,
                      size_t n, int begin_bit, int end_bit, SortScratch& scratch);

// Keys per thread of a 256-thread tile.  A tile's keys are ranked 256 at a
// time, one round after the other (about 1 us each), so few keys want small
// tiles: a scatter of 20,000 pairs took 16 us with 16 rounds, 7 us with 4;
// from 2^17 pairs on, 16 rounds fill the chip and keep the histogram (256
// entries per tile, scanned by one work-group) short.
constexpr size_t kRadix = 256, kSmallTileMax = (size_t)1 << 17;
constexpr size_t radix_items(size_t n) { return n <= kSmallTileMax ? 4 : 16; }
constexpr size_t radix_tiles(size_t n) { return (n + kRadix * radix_items(n) - 1) / (kRadix * radix_items(n)); }
// Histogram entries that sorts of up to n pairs need.
constexpr size_t radix_hist_entries(size_t n) {
  const size_t a = radix_tiles(n), b = radix_tiles(n < kSmallTileMax ? n : kSmallTileMax);
  return kRadix * (a > b ? a : b);
}

}  // namespace cloth
