// How a short reduction hands a workgroup's partial to its last workgroup.
// Plain C++ apart from the function qualifiers; Mem does the memory accesses
// (agent-scope atomics on the device).
#pragma once

namespace rpx {

// A slot is two 64-bit words, zero between calls, each 32 bits of the partial
// under a mark.  slot_take's wait is bounded, and a writer that comes after it
// gave up finds kSlotGivenUp in the words and zeroes them again, so every slot
// is zero once the launch has ended, whatever happened in it: a partial left
// standing would be taken for the next call's.
constexpr unsigned long long kSlotMark = 1ull << 32, kSlotGivenUp = 1ull << 33;

// By the one writer of slot s.
template <class Mem>
__host__ __device__ inline void slot_leave(unsigned long long* s, unsigned long long bits) {
  const unsigned long long a = Mem::exchange(s, kSlotMark | bits >> 32);
  const unsigned long long b = Mem::exchange(s + 1, kSlotMark | (bits & 0xFFFFFFFFull));
  if (a == kSlotGivenUp) Mem::store(s, 0ull);
  if (b == kSlotGivenUp) Mem::store(s + 1, 0ull);
}

// By its one reader: true and the partial, or false after `limit` fruitless looks.
template <class Mem>
__host__ __device__ inline bool slot_take(unsigned long long* s, unsigned limit, unsigned long long* bits) {
  unsigned long long hi, lo;
  for (unsigned looks = 0;;) {
    hi = Mem::load(s);
    lo = Mem::load(s + 1);
    if ((hi & lo & kSlotMark) != 0) {
      Mem::store(s, 0ull);
      Mem::store(s + 1, 0ull);
      break;
    }
    if (++looks > limit) {
      hi = Mem::exchange(s, kSlotGivenUp);
      lo = Mem::exchange(s + 1, kSlotGivenUp);
      if ((hi & kSlotMark) != 0) Mem::store(s, 0ull);
      if ((lo & kSlotMark) != 0) Mem::store(s + 1, 0ull);
      if ((hi & lo & kSlotMark) == 0) return false;
      break;
    }
    Mem::pause();
  }
  *bits = hi << 32 | (lo & 0xFFFFFFFFull);
  return true;
}

}  // namespace rpx
