// SCAN's look-back words and the segment tables that may lie where a later
// call keeps its words.  Plain C++ apart from the function qualifiers.
#pragma once

#include <stdint.h>

namespace rpx {

// A published look-back word is epoch << 24 | status << 22 | 22 bits of value
// (or of nothing), status 1 or 2.  Epochs are taken modulo 2^40.
__host__ __device__ inline unsigned long long tile_tag(unsigned long long epoch, unsigned status) {
  return (epoch << 2 | status) << 22;
}
// The status that `word` gives its tile in this epoch, 0 if none.
__host__ __device__ inline unsigned tile_status(unsigned long long word, unsigned long long epoch) {
  const unsigned long long tag = word >> 22;
  return tag >> 2 == epoch ? unsigned(tag & 3) : 0;
}

// The segmented form keeps its tables behind its words, where a single-array
// call with more tiles on the same scratch has words of its own: a bare
// element offset from 5 * 2^22 up would be the status of an early epoch there.
// Every 64 bits of the tables have the top bit set, which is that of epochs
// from 2^39 up, so none is a status that a look-back will accept.  A tile's
// segment takes half of 64 bits, and the table a whole number of them.
__host__ __device__ inline uint64_t table_entry(int64_t v) { return uint64_t(v) | uint64_t(1) << 63; }
__host__ __device__ inline int64_t table_value(uint64_t e) { return int64_t(e & ~(uint64_t(1) << 63)); }
__host__ __device__ inline uint32_t segment_entry(int s) { return uint32_t(s) | uint32_t(1) << 31; }
__host__ __device__ inline int segment_value(uint32_t e) { return int(e & ~(uint32_t(1) << 31)); }

}  // namespace rpx
