// SORT: segmented ascending sort of FP64 keys, in place.
//
// Reference: src/algorithm/SORT.hpp:18-25 (rep irep sorts the length-N
// segment x + irep*N), SORT-Seq.cpp:31-42 (std::sort), SORT-Hip.cpp:35-43
// (RAJA::sort on the device; the suite has no hand-written GPU sort).
//
// Keys are ordered by the 64-bit image of the double (sign bit set for
// non-negative values, all bits flipped for negative ones), whose unsigned
// order is numeric order with -0.0 before +0.0 and NaNs at the ends.  Equal
// images are equal bit patterns, so the sort need not be stable.
//
// MI355X design: a sample sort.  A bucket of up to 7664 keys is sorted in
// registers and LDS by one workgroup (bucket_kernel); a longer segment is
// first cut into buckets of about 4000 keys by splitters taken from a sorted
// random sample of it:
//   sample:  one workgroup per segment sorts a sample, writes the splitters;
//   hist:    every key's bucket (search over the splitters in LDS), kept as
//            16 bits, and the bucket counts of each row of 4096-key tiles;
//   colscan: each bucket's counts, scanned over the segment's rows;
//   scatter: keys to their buckets, each tile grouped by bucket in LDS first;
//   bucket:  every bucket (and every short segment) sorted.
// So a key moves twice and is read once more, where a least-significant-digit
// radix sort of 8-bit digits, which this replaces, moves it eight times and
// reads it eight times more: 41.6 M keys in 256 ragged segments 2.30 -> 0.58
// ms, one segment of 10^6 keys (24 launches then, 7 now) 0.30 -> 0.054 ms.
// Segments above kOneLevel keys are cut twice, first into about
// sqrt(n / 4096) parts.  Keys equal to a repeated splitter go round robin to
// the buckets between its copies, which hold nothing else and are not sorted,
// so equal keys cannot overfill a bucket.  A bucket that is overfull by bad
// luck in the sample is sorted in pieces that are then merged (overfull_kernel).
#include <algorithm>
#include <vector>

#include "rpx_common.hpp"

using namespace rpx;

namespace {

typedef unsigned long long u64;

// Work-items of hist and scatter, eight keys each.  What bounds both is the
// latency of their LDS phases and loads; with 256 work-items of 16 keys half as
// many wavefronts fit on a CU, and hist took 150 us instead of 101 (41.6 M keys).
constexpr int kBS = 512;
constexpr int kRows = 8;
constexpr int kTile = kBS * kRows;  // 4096 keys per tile of hist and scatter
constexpr int kAim = 4096;          // least mean of keys per bucket
constexpr int kMaxK = 1024;         // buckets per segment and level
constexpr int kCol = 64;            // buckets per workgroup of colscan
// Longest segment cut in one level: 512 buckets leave runs of 8 keys (64
// bytes) per tile and bucket to write.
constexpr long long kOneLevel = 512ll * kAim;

// A bucket_kernel workgroup of 2^TB work-items: the keys it sorts, and its
// LDS, of which sixteen wavefronts' fit on a CU (__syncthreads_or takes 256
// bytes besides).
template <int TB>
struct Room {
  static constexpr int kT = 1 << TB, kCap = 15 * kT - 16;
  static constexpr int kBytes = 160 * kT - 256;
};
constexpr int kTB = 9;  // the workgroups of long segments
typedef Room<kTB> Large;
typedef Room<8> Small;

// A segment at one level: keys [base, base + len) of x (src = 0) or of the
// scratch copy (src = 1; both are indexed alike), cut into k buckets that
// go to the other of the two.  k = 1: left where it is.
struct Seg {
  long long base, count_base;  // first key; first entry in the count table
  int len, k, rows, first_row, first_bucket, first_col;
  int src, pure;  // pure: all keys equal
};

// Number of rows, buckets and column groups of a level whose segments were
// found on the device, and of the overfull buckets.
struct Header {
  int rows, buckets, cols, over;
};

// One level.  segs = null: nseg segments of equal length from x[0], all
// alike (`one` describes the first).
struct Level {
  const Seg* segs;
  Seg one;
  int nseg;
  int chunk;  // tiles per row
  const Header* bound;  // device counts, or null where the grid is exact
  int* row_seg;
  int* col_seg;
  int* bucket_seg;   // null where every segment is one bucket
  int* dup;          // per segment: a splitter is repeated
  u64* splitters;    // [first_bucket + j], j < k - 1, ascending
  unsigned* counts;  // [count_base + row * k + bucket]
  unsigned* totals;  // [first_bucket + bucket]
  unsigned* starts;  // first key of the bucket in its segment; top bit: pure
  unsigned short* ids;
  Header* header;
  int* over;  // overfull buckets
};

__device__ __forceinline__ u64 to_key(u64 b) { return (b >> 63) ? ~b : (b | 0x8000000000000000ull); }
__device__ __forceinline__ u64 from_key(u64 u) { return (u >> 63) ? (u & 0x7FFFFFFFFFFFFFFFull) : ~u; }

__device__ __forceinline__ Seg get_seg(const Level& l, int s) {
  if (l.segs) return l.segs[s];
  Seg g = l.one;
  g.base = (long long)s * g.len;
  g.count_base = (long long)s * g.rows * g.k;
  g.first_row = s * g.rows;
  g.first_bucket = s * g.k;
  g.first_col = s * ((g.k + kCol - 1) / kCol);
  return g;
}

// Sampled keys for a cut into k buckets.  A bucket's share has a spread of
// sqrt(k / samples) of its mean, and may be 4.5 of those above it before it is
// overfull: with kAim in place of this rule, buckets of 41.6 M keys in 256
// segments were half as full and took 237 us in
// bucket_kernel instead of 212.
__host__ __device__ constexpr int samples_for(int k) { return k <= 16 ? 2048 : 8192; }
__host__ __device__ inline int buckets_for(long long len, bool whole) {
  if (len <= Large::kCap) return 1;
  if (whole || len <= kOneLevel) {
    long long k = (len + kAim - 1) / kAim;
    if (k >= kMaxK) return kMaxK;
    for (int i = 0; i < 3; ++i) {
      const float spread = sqrtf(float(k) / float(samples_for(int(k))));
      const long long aim = (long long)(float(Large::kCap) / (1.0f + 4.5f * spread));
      if (aim > kAim) k = (len + aim - 1) / aim;
    }
    return int(k < 2 ? 2 : k);
  }
  // Two levels: about sqrt(len / kAim) parts each.
  int k = 2;
  while ((long long)k * k * kAim < len && k < kMaxK) ++k;
  return k;
}

// ---- sorting network in registers and LDS ------------------------------------
//
// Where the linear map below does not do: 2^TB work-items sort N = 2^M keys
// (M = TB + RB, R = 2^RB per work-item) with a bitonic network whose merges
// begin with the mirrored comparison (i with i ^ (2^k - 1)), so every
// comparison is ascending.  A
// work-item holds the R keys whose indexes differ in bits [LO, LO + RB) and
// runs up to RB strides on registers before the keys change places through
// LDS; element i lives at LDS slot i + i/R, which spreads every layout over
// the banks.  A work-item writes only slots that it has itself just read, so
// one barrier per exchange is enough, and none (an in-order LDS queue) while
// the merged runs lie within one wavefront's 64 R keys.
//
// What bounds it: 1 VALU operation per key and stage (78 stages for 4096
// keys) and 2 ceil(k/RB) LDS accesses per key and merge.  Keys are compared as
// doubles, with one v_min_f64 and one v_max_f64 per pair where the integer
// images would take a 64-bit compare and four selects: a negative double's
// bit pattern is incremented first, which keeps the order, takes -0.0 away
// from +0.0, and leaves out only NaNs and -inf.  A workgroup that holds one of
// those first moves all images by the same amount into the range without them
// (image_shift), or, where they span more than that, sorts the images: 10^5
// keys, 100 of them NaN, take 75 us so, 142 with the images, and 132 took the
// radix sort that did not mind.  (The instructions are written out because
// fmin/fmax quieten each operand with an extra v_max_f64 when it comes from LDS.)
struct AsDouble {
  typedef double T;
  static __device__ __forceinline__ void order(double& a, double& b) {
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
  }
  static __device__ __forceinline__ double enter(u64 b) { return __longlong_as_double((long long)(b + (b >> 63))); }
  static __device__ __forceinline__ u64 leave(double d) {
    const u64 b = (u64)__double_as_longlong(d);
    return b - (b >> 63);
  }
  static __device__ __forceinline__ double last() { return __longlong_as_double(0x7FF0000000000000ll); }
};
struct AsImage {
  typedef u64 T;
  static __device__ __forceinline__ void order(u64& a, u64& b) {
    const bool swap = b < a;
    const u64 lo = swap ? b : a, hi = swap ? a : b;
    a = lo;
    b = hi;
  }
  static __device__ __forceinline__ u64 enter(u64 b) { return to_key(b); }
  static __device__ __forceinline__ u64 leave(u64 u) { return from_key(u); }
  static __device__ __forceinline__ u64 last() { return ~0ull; }
};
// Bits of a key whose image is moved up by `shift`, and back.
__device__ __forceinline__ u64 shifted(u64 b, u64 shift) { return from_key(to_key(b) + shift); }
__device__ __forceinline__ u64 unshifted(u64 b, u64 shift) { return from_key(to_key(b) - shift); }
// Looks the images of keys get(0) .. get(len - 1) over.  *shift takes the least
// to the least that AsDouble orders, -DBL_MAX's; false, and no shift, where the
// greatest would then be above +inf's.  Ends with `mem` free.
template <int kT, class Get>
__device__ __forceinline__ bool image_shift(int len, Get get, char* mem, int t, u64* shift) {
  constexpr int kWaves = kT / kWave;
  constexpr u64 kLeast = 0x0010000000000000ull, kMost = 0xFFF0000000000000ull;
  u64* ends = reinterpret_cast<u64*>(mem);
  u64 lo = ~0ull, hi = 0ull;
  for (int i = t; i < len; i += kT) {
    const u64 k = to_key(get(i));
    lo = k < lo ? k : lo;
    hi = k > hi ? k : hi;
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const u64 l = __shfl_xor(lo, off, kWave), h = __shfl_xor(hi, off, kWave);
    lo = l < lo ? l : lo;
    hi = h > hi ? h : hi;
  }
  if (t % kWave == 0) {
    ends[t / kWave] = lo;
    ends[kWaves + t / kWave] = hi;
  }
  __syncthreads();
  for (int w = 0; w < kWaves; ++w) {
    lo = ends[w] < lo ? ends[w] : lo;
    hi = ends[kWaves + w] > hi ? ends[kWaves + w] : hi;
  }
  __syncthreads();
  const bool fits = __builtin_amdgcn_readfirstlane(hi - lo <= kMost - kLeast) != 0;  // the same in all lanes
  const u64 s = fits ? kLeast - lo : 0ull;
  *shift = u64(unsigned(__builtin_amdgcn_readfirstlane(int(s >> 32)))) << 32 |
           unsigned(__builtin_amdgcn_readfirstlane(int(s)));
  return fits;
}

template <class C, int TB, int RB>
struct Net {
  typedef typename C::T T;
  static constexpr int kT = 1 << TB, R = 1 << RB, M = TB + RB, N = 1 << M;
  static constexpr int kSlots = N + N / R;

  // LDS slot of element (hi, r, lo) of layout LO is base + offset(r).
  template <int LO>
  static __device__ __forceinline__ int base(int t, bool flip) {
    const int mask = (1 << LO) - 1;
    const int lo = (flip ? ~t : t) & mask;
    const int i = ((t >> LO) << (LO + RB)) | lo;
    return i + (i >> RB);
  }
  template <int LO>
  static __device__ __forceinline__ constexpr int offset(int r) {
    return (r << LO) + ((r << LO) >> RB);
  }
  // In layout LO > 0 of a merge's first exchange the upper half of the
  // registers holds elements whose low index bits are complemented.
  template <int LO, bool FLIP>
  static __device__ __forceinline__ void get(T (&v)[R], const T* lds, int t) {
    const int b0 = base<LO>(t, false), b1 = FLIP ? base<LO>(t, true) : b0;
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = lds[(r < R / 2 ? b0 : b1) + offset<LO>(r)];
  }
  template <int LO, bool FLIP>
  static __device__ __forceinline__ void put(const T (&v)[R], T* lds, int t) {
    const int b0 = base<LO>(t, false), b1 = FLIP ? base<LO>(t, true) : b0;
#pragma unroll
    for (int r = 0; r < R; ++r) lds[(r < R / 2 ? b0 : b1) + offset<LO>(r)] = v[r];
  }
  // Strides 2^S .. 1 of the register index.
  template <int S>
  static __device__ __forceinline__ void strides(T (&v)[R]) {
    if constexpr (S >= 0) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if ((r & (1 << S)) == 0) C::order(v[r], v[r | (1 << S)]);
      strides<S - 1>(v);
    }
  }
  template <int K>
  static __device__ __forceinline__ void mirror(T (&v)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if ((r & (1 << (K - 1))) == 0) C::order(v[r], v[r ^ ((1 << K) - 1)]);
  }
  template <int K>
  static __device__ __forceinline__ void exchange_sync() {
    if constexpr (K > 6 + RB) __syncthreads();
    else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  // The strides of merge K below layout HI's, down to layout 0.
  template <int K, int HI>
  static __device__ __forceinline__ void descend(T (&v)[R], T* lds, int t) {
    if constexpr (HI > 0) {
      constexpr int LO = HI > RB ? HI - RB : 0;
      exchange_sync<K>();
      get<LO, false>(v, lds, t);
      strides<HI - 1 - LO>(v);
      if constexpr (LO > 0) put<LO, false>(v, lds, t);
      descend<K, LO>(v, lds, t);
    }
  }
  template <int K>
  static __device__ __forceinline__ void merges(T (&v)[R], T* lds, int t) {
    if constexpr (K <= RB) {
      mirror<K>(v);
      strides<K - 2>(v);
      merges<K + 1>(v, lds, t);
    } else if constexpr (K <= M) {
      constexpr int LO = K - RB;
      put<0, false>(v, lds, t);
      exchange_sync<K>();
      get<LO, true>(v, lds, t);
      mirror<RB>(v);
      strides<RB - 2>(v);
      put<LO, true>(v, lds, t);
      descend<K, LO>(v, lds, t);
      merges<K + 1>(v, lds, t);
    }
  }
  // v in any order -> v[r] = element R t + r of the sorted sequence; lds
  // (kSlots values) is overwritten.
  static __device__ __forceinline__ void sort(T (&v)[R], T* lds, int t) { merges<1>(v, lds, t); }

  // Sorts the keys b, key r of work-item t being key r kT + t, into dst, len <= N;
  // they come shifted and leave as they were.
  static __device__ __forceinline__ void sort_keys(const u64 (&b)[R], u64 shift, u64* dst, int len, void* mem, int t) {
    T* lds = reinterpret_cast<T*>(mem);
    T v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = (r * kT + t < len) ? C::enter(b[r]) : C::last();
    sort(v, lds, t);
    put<0, false>(v, lds, t);
    __syncthreads();
    const auto store = [&](auto leave) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int i = r * kT + t;
        if (i < len) dst[i] = leave(lds[i + (i >> RB)]);
      }
    };
    if (shift == 0) store([](T v) { return C::leave(v); });
    else store([&](T v) { return unshifted(C::leave(v), shift); });
  }
};

// ---- sorting by a linear map --------------------------------------------------
//
// The keys of a bucket lie between two neighbouring splitters, where most
// inputs are close to evenly spread.  2^TB work-items map up to 16 keys each
// onto 16 bins each, linearly from the least key to the greatest, count the
// bins with LDS atomics (a counter's old value is the key's place in its bin)
// and put the keys into their bins' slots.  The map is monotone in floating
// point, so only keys of one bin can be out of order.  A work-item then sorts
// 16 consecutive slots in registers and merges its upper eight with its
// neighbour's lower eight, which sorts all if no bin holds more than nine
// different keys; half a key per bin is usual.  Whether it did is read off the
// neighbours of the merged sixteens.  If not, or with NaNs, infinities, or a
// -0.0 (which equals +0.0 as a double), nothing has been written and the
// network sorts the keys.
//
// What bounds it: about 50 vector instructions and 60 bytes of LDS traffic per
// key, where the network spends 91 comparisons and 360 bytes; each takes 40% of
// the time, as do the 16 bytes per key from and to memory, and the eight
// barriers between them keep a workgroup waiting.  Buckets of 41.6 M keys: 407
// us with the network alone (4096 keys at most, the overfull in a kernel of 52
// us), 212 us here.  Ranking the keys of a bin by comparing each with all
// others took 315 us.
// Odd-even merges of sorted runs of P keys into longer ones, up to all 16.
template <int P, int K = P>
__device__ __forceinline__ void batcher(double (&v)[16]) {
#pragma unroll
  for (int i = 0; i < 16 - K; ++i)
    if (i >= K % P && (i - K % P) / K % 2 == 0 && i / (2 * P) == (i + K) / (2 * P)) AsDouble::order(v[i], v[i + K]);
  if constexpr (K > 1) batcher<P, K / 2>(v);
  else if constexpr (P < 8) batcher<2 * P>(v);
}

// Exclusive scan over the work-items of a workgroup (one value each).
__device__ __forceinline__ unsigned block_exclusive_scan(unsigned v, unsigned* wsum) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  unsigned incl = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const unsigned o = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += o;
  }
  if (lane == kWave - 1) wsum[wave] = incl;
  __syncthreads();
  unsigned run = incl - v;
  for (int w = 0; w < wave; ++w) run += wsum[w];
  return run;
}

// LDS of up to `keys` keys: 17 words per 16 of them (both a work-item's 16 and
// adjacent work-items' keys then fall into different banks), and the bins.
constexpr int linear_bytes(int tb, int keys) { return keys / 16 * 17 * 8 + (32 << tb); }
static_assert(linear_bytes(kTB, Large::kCap) <= Large::kBytes && linear_bytes(8, Small::kCap) <= Small::kBytes &&
                  Large::kCap % 16 == 0 && Small::kCap % 16 == 0,
              "keys and bins fit");

// get(i): the bits of key i, 0 <= i < len, 1 <= len <= kKeys <= 2^(TB+4).
// Calls out(place, key) for every key, or says why not, by all work-items.
enum Linear { kSorted, kUneven, kSpecial };  // kSpecial: with a NaN or an infinity
template <int TB, int kKeys, class Get, class Out>
__device__ __forceinline__ Linear sort_linear(int len, char* lds, int t, Get get, Out out) {
  constexpr int T = 1 << TB, R = 16, N = T * R, kWaves = T / kWave, W = R / 2;
  static_assert(kKeys <= N && kKeys % 16 == 0 && N <= 65536, "16-bit counters");
  double* keys = reinterpret_cast<double*>(lds);
  unsigned* bins = reinterpret_cast<unsigned*>(lds + kKeys / 16 * 17 * 8);  // two 16-bit counters per word
  double* ends = keys;                                                      // before any key is placed
  unsigned* wsum = reinterpret_cast<unsigned*>(ends + 2 * kWaves);
  const int lane = t & (kWave - 1), wave = t / kWave;
  auto slot = [](int i) { return i + (i >> 4); };
  double x[R];
  unsigned widest = 0u;
  bool special = false;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = (r << TB) + t;
    if ((r << TB) < len) x[r] = __longlong_as_double((long long)get(i < len ? i : len - 1));
  }
#pragma unroll
  for (int j = 0; j < W; ++j) bins[j * T + t] = 0u;
  double lo = x[0], hi = x[0];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if ((r << TB) >= len) continue;
    const u64 b = (u64)__double_as_longlong(x[r]);
    const unsigned size = unsigned(b >> 32) & 0x7FFFFFFFu;
    widest = size > widest ? size : widest;
    special |= b == 0x8000000000000000ull;
    asm("v_min_f64 %0, %0, %1" : "+v"(lo) : "v"(x[r]));
    asm("v_max_f64 %0, %0, %1" : "+v"(hi) : "v"(x[r]));
  }
  const bool wide = widest >= 0x7FF00000u;
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const double l = __shfl_xor(lo, off, kWave), h = __shfl_xor(hi, off, kWave);
    asm("v_min_f64 %0, %0, %1" : "+v"(lo) : "v"(l));
    asm("v_max_f64 %0, %0, %1" : "+v"(hi) : "v"(h));
  }
  if (lane == 0) {
    ends[wave] = lo;
    ends[kWaves + wave] = hi;
  }
  if (__syncthreads_or(special || wide)) return __syncthreads_or(wide) ? kSpecial : kUneven;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const double l = ends[w], h = ends[kWaves + w];
    asm("v_min_f64 %0, %0, %1" : "+v"(lo) : "v"(l));
    asm("v_max_f64 %0, %0, %1" : "+v"(hi) : "v"(h));
  }
  const double spread = hi - lo;
  const double scale = double(N) / spread;
  if (!(spread < 1e300 && scale < 1e300)) {
    if (spread != 0.0) return kUneven;
#pragma unroll
    for (int r = 0; r < R; ++r)  // all equal
      if ((r << TB) + t < len) out((r << TB) + t, (u64)__double_as_longlong(x[r]));
    return kSorted;
  }
  unsigned at[R];  // the key's bin, and its place in it above
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if ((r << TB) >= len) continue;
    int bin = int((x[r] - lo) * scale);
    bin = bin < N - 1 ? bin : N - 1;
    at[r] = unsigned(bin);
    if ((r << TB) + t < len) {
      const unsigned old = atomicAdd(&bins[bin >> 1], 1u << (bin << 4 & 31));
      at[r] |= old >> (bin << 4 & 31) << 16;
    }
  }
  __syncthreads();
  {
    unsigned c[W], sum = 0;
#pragma unroll
    for (int j = 0; j < W; ++j) {
      c[j] = bins[t * W + j];
      sum += (c[j] & 0xFFFFu) + (c[j] >> 16);
    }
    unsigned run = block_exclusive_scan(sum, wsum);
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const unsigned second = run + (c[j] & 0xFFFFu);
      bins[t * W + j] = run | second << 16;
      run = second + (c[j] >> 16);
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if ((r << TB) + t < len) {
      const unsigned bin = at[r] & 0xFFFFu;
      keys[slot(int((bins[bin >> 1] >> (bin << 4 & 31) & 0xFFFFu) + (at[r] >> 16)))] = x[r];
    }
  }
  __syncthreads();
  const double none = __longlong_as_double(0x7FF0000000000000ll);
  const int first = 16 * t;
  double* own = keys + 17 * t;  // slots first .. first + 15; the next work-item's from own + 17
  if (first < len) {
#pragma unroll
    for (int u = 0; u < 16; ++u) x[u] = own[u];
    if (first + 16 > len) {
#pragma unroll
      for (int u = 0; u < 16; ++u) x[u] = first + u < len ? x[u] : none;
    }
    batcher<1>(x);
#pragma unroll
    for (int u = 0; u < 8; ++u) own[u] = x[u];
  }
  __syncthreads();
  if (first + 8 < len) {
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = x[u + 8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u + 8] = first + 16 < len ? own[17 + u] : none;
    batcher<8>(x);
#pragma unroll
    for (int u = 0; u < 8; ++u) own[8 + u] = x[u];
    if (first + 16 < len) {
#pragma unroll
      for (int u = 0; u < 8; ++u) own[17 + u] = x[u + 8];
    }
  }
  __syncthreads();
  bool bad = t == 0 && len > 8 && keys[7] > keys[8];
  if (first + 24 < len) bad |= own[17 + 7] > own[17 + 8];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if ((r << TB) + t < len) x[r] = keys[slot((r << TB) + t)];
  }
  if (__syncthreads_or(bad)) return kUneven;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if ((r << TB) + t < len) out((r << TB) + t, (u64)__double_as_longlong(x[r]));
  }
  return kSorted;
}

template <int TB, int RB>
__device__ __forceinline__ void sort_network(const u64* src, u64* dst, int len, bool doubles, u64 shift, char* lds,
                                             int t) {
  u64 b[1 << RB];
#pragma unroll
  for (int r = 0; r < (1 << RB); ++r) {
    const int i = (r << TB) + t;
    b[r] = i < len ? src[i] : 0ull;
  }
  if (shift != 0) {
#pragma unroll
    for (int r = 0; r < (1 << RB); ++r) b[r] = shifted(b[r], shift);
  }
  if (doubles) Net<AsDouble, TB, RB>::sort_keys(b, shift, dst, len, lds, t);
  else Net<AsImage, TB, RB>::sort_keys(b, shift, dst, len, lds, t);
}

static_assert(Net<AsDouble, kTB, 4>::kSlots * 8 <= Large::kBytes && Net<AsDouble, 8, 4>::kSlots * 8 <= Small::kBytes,
              "the networks fit too");

// src[0..len) -> dst sorted (dst may be src), 1 <= len <= Room<TB>::kCap.
template <int TB>
__device__ __forceinline__ void sort_piece(const u64* src, u64* dst, int len, char* lds, int t) {
  // 32-bit byte offsets from a uniform base
  const auto get = [&](int i) {
    return *reinterpret_cast<const u64*>(reinterpret_cast<const char*>(src) + unsigned(i) * 8u);
  };
  const auto put = [&](int i, u64 v) {
    *reinterpret_cast<u64*>(reinterpret_cast<char*>(dst) + unsigned(i) * 8u) = v;
  };
  const Linear done = sort_linear<TB, Room<TB>::kCap>(len, lds, t, get, put);
  if (done == kSorted) return;
  __syncthreads();
  u64 shift = 0;
  const bool doubles = done != kSpecial || image_shift<1 << TB>(len, get, lds, t, &shift);
  if (len <= 4 << TB) sort_network<TB, 2>(src, dst, len, doubles, shift, lds, t);
  else sort_network<TB, 4>(src, dst, len, doubles, shift, lds, t);
}

// ---- splitters -----------------------------------------------------------------

// Sample of segment s, sorted, and every k-quantile of it as a splitter.
// S = 2^(kTB+RB) keys from S equal strata at pseudo-random places in them.
template <class C, int RB>
__device__ __forceinline__ void network_splitters(const u64 (&b)[1 << RB], u64 shift, int k, u64* sp, char* mem,
                                                  int t) {
  typedef Net<C, kTB, RB> W;
  typename C::T* lds = reinterpret_cast<typename C::T*>(mem);
  typename C::T v[W::R];
#pragma unroll
  for (int r = 0; r < W::R; ++r) v[r] = C::enter(b[r]);
  W::sort(v, lds, t);
  W::template put<0, false>(v, lds, t);
  __syncthreads();
  for (int j = t + 1; j < k; j += W::kT) {
    const int i = j * W::N / k;  // j < 1024
    sp[j - 1] = to_key(C::leave(lds[i + (i >> RB)])) - shift;
  }
}

// Key i of the 2^m sampled from len at src: that at (i + jitter 2^-16) len / 2^m.
__device__ __forceinline__ u64 sampled_key(const u64* src, int len, int i, int m) {
  const u64 jitter = mix64(u64(i) * kGamma + u64(len)) >> 48;
  return src[(u64(i) << 16 | jitter) * u64(len) >> (16 + m)];
}

// A CU takes about 20 us to read 8192 keys from as many lines.  Where the
// segments leave CUs free, kGather of them read a segment's sample and leave it
// side by side where the segment's keys will go (10^6 keys: 28 us -> 5 and 10).
constexpr int kGather = 8, kGatherSegs = 128;
__global__ __launch_bounds__(256) void gather_kernel(u64* x, u64* alt, Level l) {
  const int s = blockIdx.x / kGather;
  const Seg g = get_seg(l, s);
  if (g.k <= 1) return;
  const u64* src = (g.src ? alt : x) + g.base;
  u64* dst = (g.src ? x : alt) + g.base;
  const int m = samples_for(g.k) == 2048 ? 11 : 13;
  for (int i = int(blockIdx.x) % kGather * 256 + int(threadIdx.x); i < 1 << m; i += kGather * 256)
    dst[i] = sampled_key(src, g.len, i, m);
}

template <int RB>
__device__ __forceinline__ void sample_segment(const u64* src, bool gathered, const Seg& g, u64* splitters, int* dup,
                                               u64* sp, char* mem, int t) {
  constexpr int R = 1 << RB, T = 1 << kTB, M = kTB + RB, S = 1 << M;
  const auto sampled = [&](int i) { return gathered ? src[i] : sampled_key(src, g.len, i, M); };
  // Quantile j is the key at place floor(j S / k).
  const auto quantile = [&](int place, u64 b) {
    const int j = int((unsigned(place) * unsigned(g.k) + unsigned(S - 1)) >> M);
    if (j > 0 && j < g.k && (unsigned(j) << M) < unsigned(place + 1) * unsigned(g.k)) sp[j - 1] = to_key(b);
  };
  if (const Linear done = sort_linear<kTB, S>(S, mem, t, sampled, quantile); done != kSorted) {
    __syncthreads();
    u64 shift = 0;
    const bool doubles = done != kSpecial || image_shift<T>(S, sampled, mem, t, &shift);
    u64 b[R];
#pragma unroll
    for (int r = 0; r < R; ++r) b[r] = shifted(sampled(r * T + t), shift);
    if (doubles) network_splitters<AsDouble, RB>(b, shift, g.k, sp, mem, t);
    else network_splitters<AsImage, RB>(b, shift, g.k, sp, mem, t);
  }
  __syncthreads();
  bool d = false;
  for (int j = t; j < g.k - 1; j += T) {
    splitters[j] = sp[j];
    d |= j > 0 && sp[j] == sp[j - 1];
  }
  const int any = __syncthreads_or(d);
  if (t == 0) *dup = any;
}

// One workgroup per segment: its entries of the row, column and bucket maps,
// and its splitters.
constexpr int kSampleBytes = linear_bytes(kTB, 8192);
static_assert(kSampleBytes >= 8 * Net<AsDouble, kTB, 4>::kSlots, "the network fits too");
__global__ __launch_bounds__(1 << kTB) void sample_kernel(const u64* x, const u64* alt, Level l, bool gathered) {
  __shared__ __attribute__((aligned(16))) char mem[kSampleBytes];
  __shared__ u64 sp[kMaxK];
  constexpr int T = 1 << kTB;
  const int t = threadIdx.x, s = blockIdx.x;
  if (s == 0 && t == 0) l.header->over = 0;
  const Seg g = get_seg(l, s);
  if (l.segs) {
    for (int i = t; i < g.k; i += T) l.bucket_seg[g.first_bucket + i] = s;
    if (g.k > 1) {
      for (int i = t; i < g.rows; i += T) l.row_seg[g.first_row + i] = s;
      for (int i = t; i < (g.k + kCol - 1) / kCol; i += T) l.col_seg[g.first_col + i] = s;
    }
  }
  if (g.k <= 1) return;
  const u64* src = ((g.src != 0) != gathered ? alt : x) + g.base;
  u64* splitters = l.splitters + g.first_bucket;
  if (samples_for(g.k) == 2048) sample_segment<2>(src, gathered, g, splitters, l.dup + s, sp, mem, t);
  else sample_segment<4>(src, gathered, g, splitters, l.dup + s, sp, mem, t);
}

// ---- partition -----------------------------------------------------------------

// Segment of row, column group or bucket i.
__device__ __forceinline__ int seg_of(const Level& l, const int* map, int i, int per_seg) {
  if (!l.segs) return i / per_seg;
  return map ? map[i] : i;
}

// A row is `chunk` tiles.  The search runs over the splitters as a complete
// binary tree in breadth-first order (missing ones above every key): a
// level's nodes lie together, so the top five levels are free of bank
// conflicts.
__global__ __launch_bounds__(kBS) void hist_kernel(const u64* x, const u64* alt, Level l) {
  __shared__ u64 tree[kMaxK];
  __shared__ u64 sorted[kMaxK];
  __shared__ unsigned cnt[kMaxK];
  const int t = threadIdx.x;
  const int row = int(xcd_major(blockIdx.x, gridDim.x));
  if (l.bound && row >= l.bound->rows) return;
  const int s = seg_of(l, l.row_seg, row, l.one.rows);
  const Seg g = get_seg(l, s);
  int depth = 1;
  while ((1 << depth) < g.k) ++depth;
  const u64* sp = l.splitters + g.first_bucket;
  for (int j = t; j < (1 << depth); j += kBS) {
    const u64 v = j < g.k - 1 ? sp[j] : ~0ull;
    sorted[j] = v;
    cnt[j] = 0u;
    const int z = __ffs(j + 1) - 1;  // node of rank j: 2^z divides j + 1
    if (j + 1 < (1 << depth)) tree[(1 << (depth - 1 - z)) - 1 + ((j + 1) >> (z + 1))] = v;
  }
  const bool dup = l.dup[s] != 0;
  __syncthreads();
  const long long local0 = (long long)(row - g.first_row) * l.chunk * kTile;
  const u64* src = (g.src ? alt : x) + g.base;
  unsigned short* ids = l.ids + g.base;
  for (int c = 0; c < l.chunk; ++c) {
    const long long first = local0 + (long long)c * kTile;
    if (first >= g.len) break;
    const int n = int(g.len - first < kTile ? g.len - first : kTile);
    u64 k[kRows];
    int node[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int i = r * kBS + t;
      k[r] = i < n ? to_key(src[first + i]) : 0ull;
      node[r] = 0;
    }
    for (int d = 0; d < depth; ++d) {
#pragma unroll
      for (int r = 0; r < kRows; ++r) node[r] = 2 * node[r] + 1 + (tree[node[r]] < k[r] ? 1 : 0);
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int i = r * kBS + t;
      int b = node[r] - ((1 << depth) - 1);  // splitters below the key: at most k - 1
      if (dup && b < g.k - 1 && sorted[b] == k[r]) {
        // Equal to splitters b .. b + run - 1: any bucket b .. b + run will
        // do; between two copies it holds this value only.
        int lo = b + 1, hi = g.k - 1;  // the first splitter above the key
        while (lo < hi) {
          const int m = (lo + hi) >> 1;
          if (sorted[m] == k[r]) lo = m + 1;
          else hi = m;
        }
        const int run = lo - b;
        const unsigned h = unsigned(mix64(u64(first + i) * kGamma) >> 32);
        b += run == 1 ? int(h & 1u) : 1 + int((u64(h) * unsigned(run - 1)) >> 32);
      }
      if (i < n) {
        atomicAdd(&cnt[b], 1u);
        ids[first + i] = (unsigned short)b;
      }
    }
  }
  __syncthreads();
  unsigned* out = l.counts + g.count_base + (long long)(row - g.first_row) * g.k;
  for (int j = t; j < g.k; j += kBS) out[j] = cnt[j];
}

// kCol buckets of one segment: exclusive scan of their counts over the rows
// (16 walkers per bucket, each over a sixteenth of the rows), and totals.
constexpr int kWalkers = 16;
__global__ __launch_bounds__(kCol* kWalkers) void colscan_kernel(Level l) {
  __shared__ unsigned part[kWalkers][kCol];
  const int col = blockIdx.x;
  if (l.bound && col >= l.bound->cols) return;
  const int s = seg_of(l, l.col_seg, col, (l.one.k + kCol - 1) / kCol);
  const Seg g = get_seg(l, s);
  const int lane = threadIdx.x % kCol, w = threadIdx.x / kCol;
  const int b = (col - g.first_col) * kCol + lane;
  const bool live = b < g.k;
  const int q = (g.rows + kWalkers - 1) / kWalkers;
  const int r0 = w * q < g.rows ? w * q : g.rows;
  const int r1 = (w + 1) * q < g.rows ? (w + 1) * q : g.rows;
  unsigned* at = l.counts + g.count_base + b;
  constexpr int kBatch = 16;
  unsigned sum = 0;
  if (live) {
    int r = r0;
    for (; r + kBatch <= r1; r += kBatch) {
      unsigned v[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) v[u] = at[(long long)(r + u) * g.k];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) sum += v[u];
    }
    for (; r < r1; ++r) sum += at[(long long)r * g.k];
  }
  part[w][lane] = sum;
  __syncthreads();
  unsigned run = 0, total = 0;
#pragma unroll
  for (int i = 0; i < kWalkers; ++i) {
    const unsigned p = part[i][lane];
    if (i < w) run += p;
    total += p;
  }
  if (!live) return;
  if (w == 0) l.totals[g.first_bucket + b] = total;
  int r = r0;
  for (; r + kBatch <= r1; r += kBatch) {
    unsigned v[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) v[u] = at[(long long)(r + u) * g.k];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      at[(long long)(r + u) * g.k] = run;
      run += v[u];
    }
  }
  for (; r < r1; ++r) {
    const unsigned v = at[(long long)r * g.k];
    at[(long long)r * g.k] = run;
    run += v;
  }
}

// Keys of a row to their buckets.  Within a tile a key's slot is its
// bucket's first slot plus the old value of an LDS counter; the tile then
// leaves in slot order, so that each bucket's keys go to consecutive
// addresses from consecutive work-items.  Rows are numbered XCD-major: the
// partial lines at the ends of adjacent rows' runs are written from one L2.
__global__ __launch_bounds__(kBS) void scatter_kernel(u64* x, u64* alt, Level l) {
  __shared__ u64 keys[kTile];
  __shared__ unsigned short slot_id[kTile];
  __shared__ unsigned cnt[kMaxK];
  __shared__ unsigned next[kMaxK];   // where the row's next key of the bucket goes
  __shared__ unsigned delta[kMaxK];  // next - first slot
  __shared__ unsigned wsum[kBS / kWave];
  const int t = threadIdx.x;
  const int row = int(xcd_major(blockIdx.x, gridDim.x));
  if (l.bound && row >= l.bound->rows) return;
  const int s = seg_of(l, l.row_seg, row, l.one.rows);
  const Seg g = get_seg(l, s);
  const int lrow = row - g.first_row;
  constexpr int kPer = kMaxK / kBS;
  const unsigned* before = l.counts + g.count_base + (long long)lrow * g.k;
  // First key of each bucket in the segment.
  {
    unsigned tot[kPer], sum = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int b = t * kPer + j;
      tot[j] = b < g.k ? l.totals[g.first_bucket + b] : 0u;
      sum += tot[j];
    }
    unsigned run = block_exclusive_scan(sum, wsum);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int b = t * kPer + j;
      if (b < g.k) {
        next[b] = run + before[b];
        if (lrow == 0) {
          const u64* sp = l.splitters + g.first_bucket;
          const bool pure = b > 0 && b < g.k - 1 && sp[b - 1] == sp[b];
          l.starts[g.first_bucket + b] = run | (pure ? 0x80000000u : 0u);
        }
      }
      run += tot[j];
    }
  }
  const u64* src = (g.src ? alt : x) + g.base;
  u64* dst = (g.src ? x : alt) + g.base;
  const unsigned short* ids = l.ids + g.base;
  const long long local0 = (long long)lrow * l.chunk * kTile;
  for (int c = 0; c < l.chunk; ++c) {
    const long long first = local0 + (long long)c * kTile;
    if (first >= g.len) break;
    const int n = int(g.len - first < kTile ? g.len - first : kTile);
    u64 k[kRows];
    unsigned id[kRows], rank[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int i = r * kBS + t;
      id[r] = i < n ? ids[first + i] : 0u;
      k[r] = i < n ? src[first + i] : 0ull;
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) cnt[t + j * kBS] = 0u;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRows; ++r)
      if (r * kBS + t < n) rank[r] = atomicAdd(&cnt[id[r]], 1u);
    __syncthreads();
    {
      unsigned cc[kPer], sum = 0;
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        cc[j] = cnt[t * kPer + j];
        sum += cc[j];
      }
      unsigned run = block_exclusive_scan(sum, wsum);
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const int b = t * kPer + j;
        cnt[b] = run;  // first slot
        if (b < g.k) {
          delta[b] = next[b] - run;
          next[b] += cc[j];
        }
        run += cc[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRows; ++r)
      if (r * kBS + t < n) {
        const unsigned at = cnt[id[r]] + rank[r];
        keys[at] = k[r];
        slot_id[at] = (unsigned short)id[r];
      }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int i = r * kBS + t;
      if (i < n) dst[delta[slot_id[i]] + unsigned(i)] = keys[i];
    }
    __syncthreads();
  }
}

// ---- buckets -------------------------------------------------------------------

struct Piece {
  long long base;
  int len, src;
  bool pure;
};

// Bucket i of a level (a whole segment where k = 1), and where it lies.
__device__ __forceinline__ Piece get_piece(const Level& l, int i) {
  const int s = seg_of(l, l.bucket_seg, i, l.one.k);
  const Seg g = get_seg(l, s);
  if (g.k <= 1) return Piece{g.base, g.len, g.src, g.pure != 0};
  const unsigned st = l.starts[i];
  return Piece{g.base + (long long)(st & 0x7FFFFFFFu), int(l.totals[i]), 1 - g.src, (st >> 31) != 0};
}

// Any length: parts of Room<TB>::kCap keys, then merges of ever longer runs,
// every key finding its place by a search in the other run.  The parts start
// in x or alt so that the last merge ends in x.
template <int TB>
__device__ __forceinline__ void sort_any(u64* x, u64* alt, const Piece& p, char* mem, int t) {
  constexpr int kPiece = Room<TB>::kCap;
  u64* at[2] = {x + p.base, alt + p.base};
  const u64* src = at[p.src];
  int rounds = 0;
  while (((long long)kPiece << rounds) < p.len) ++rounds;
  int cur = rounds & 1;
  for (long long o = 0; o < p.len; o += kPiece) {
    const int n = int(p.len - o < kPiece ? p.len - o : kPiece);
    sort_piece<TB>(src + o, at[cur] + o, n, mem, t);
    __syncthreads();
  }
  for (long long w = kPiece; w < p.len; w *= 2) {
    const u64* a = at[cur];
    u64* d = at[cur ^ 1];
    for (long long i = t; i < p.len; i += 1 << TB) {
      const long long lo = i / (2 * w) * (2 * w);
      const long long mid = lo + w < p.len ? lo + w : p.len;
      const long long hi = lo + 2 * w < p.len ? lo + 2 * w : p.len;
      const bool left = i < mid;
      const u64 raw = a[i], key = to_key(raw);
      long long b = left ? mid : lo, e = left ? hi : mid;
      const long long b0 = b;
      while (b < e) {
        const long long m = (b + e) >> 1;
        const u64 o = to_key(a[m]);
        if (left ? o < key : o <= key) b = m + 1;
        else e = m;
      }
      d[lo + (left ? i - lo : i - mid) + (b - b0)] = raw;
    }
    __syncthreads();
    cur ^= 1;
  }
}

// Every bucket and uncut segment of up to Room<TB>::kCap keys.  Longer ones go
// on the list for overfull_kernel (in this kernel its code would spill).
template <int TB>
__global__ __launch_bounds__(1 << TB, 4) void bucket_kernel(u64* x, const u64* alt, Level l) {
  __shared__ __attribute__((aligned(16))) char mem[Room<TB>::kBytes];
  const int t = threadIdx.x, i = blockIdx.x;
  if (l.bound && i >= l.bound->buckets) return;
  const Piece p = get_piece(l, i);
  const u64* src = (p.src ? alt : x) + p.base;
  u64* dst = x + p.base;
  if (p.pure) {
    if (p.src)
      for (int j = t; j < p.len; j += 1 << TB) dst[j] = src[j];
    return;
  }
  if (p.len == 0 || (p.len == 1 && !p.src)) return;
  if (p.len <= Room<TB>::kCap) sort_piece<TB>(src, dst, p.len, mem, t);
  else if (t == 0) l.over[atomicAdd(&l.header->over, 1)] = i;
}

__global__ __launch_bounds__(1 << kTB) void overfull_kernel(u64* x, u64* alt, Level l) {
  __shared__ __attribute__((aligned(16))) char mem[Large::kBytes];
  const int n = l.header->over;
  for (int i = blockIdx.x; i < n; i += gridDim.x) {
    sort_any<kTB>(x, alt, get_piece(l, l.over[i]), mem, threadIdx.x);
    __syncthreads();
  }
}

// The second level's segments are the first level's buckets: one workgroup
// numbers their rows, buckets, column groups and count entries.
__global__ __launch_bounds__(1024) void second_level_kernel(Level l, int nbuckets, Seg* out, Header* bound, int chunk) {
  __shared__ long long sums[1024 / kWave][4];
  __shared__ long long carry[4];
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  if (t < 4) carry[t] = 0;
  __syncthreads();
  for (int i0 = 0; i0 < nbuckets; i0 += 1024) {
    const int i = i0 + t;
    Piece p{0, 0, 0, false};
    if (i < nbuckets) p = get_piece(l, i);
    Seg g;
    g.base = p.base;
    g.len = p.len;
    g.src = p.src;
    g.pure = p.pure;
    g.k = p.pure ? 1 : buckets_for(p.len, true);
    g.rows = g.k > 1 ? int((p.len + (long long)chunk * kTile - 1) / ((long long)chunk * kTile)) : 0;
    const int cols = g.k > 1 ? (g.k + kCol - 1) / kCol : 0;
    if (i >= nbuckets) g.k = 0;
    long long v[4] = {g.rows, g.k, cols, (long long)g.rows * g.k}, incl[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      incl[c] = v[c];
      for (int off = 1; off < kWave; off <<= 1) {
        const long long o = __shfl_up(incl[c], off, kWave);
        if (lane >= off) incl[c] += o;
      }
      if (lane == kWave - 1) sums[wave][c] = incl[c];
    }
    __syncthreads();
    long long first[4], total[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      first[c] = carry[c] + incl[c] - v[c];
      total[c] = carry[c];
      for (int w = 0; w < 1024 / kWave; ++w) {
        if (w < wave) first[c] += sums[w][c];
        total[c] += sums[w][c];
      }
    }
    if (i < nbuckets) {
      g.first_row = int(first[0]);
      g.first_bucket = int(first[1]);
      g.first_col = int(first[2]);
      g.count_base = first[3];
      out[i] = g;
    }
    __syncthreads();
    if (t == 0)
      for (int c = 0; c < 4; ++c) carry[c] = total[c];
    __syncthreads();
  }
  if (t == 0) {
    bound->rows = int(carry[0]);
    bound->buckets = int(carry[1]);
    bound->cols = int(carry[2]);
  }
}

inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// Sizes of one level's tables, for exact counts (first level) or bounds.
struct LevelSize {
  long long segs = 0, rows = 0, buckets = 0, cols = 0, counts = 0;
};
struct Sizes {
  long long keys = 0, longest = 0, base = 0;
  int64_t nseg = 0;  // non-empty segments
  bool uniform = true, small = true, two_levels = false;
  int chunk = 1;
  LevelSize l1, l2;
};

// Tiles per row: one, and more where that would make over 4096 rows.
int chunk_for(long long keys) {
  const long long c = keys / (4096ll * kTile);
  return int(c < 1 ? 1 : c > 64 ? 64 : c);
}

Seg describe(long long base, long long len, int chunk) {
  Seg g{};
  g.base = base;
  g.len = int(len);
  g.k = buckets_for(len, false);
  g.rows = g.k > 1 ? int(ceil_div(len, (long long)chunk * kTile)) : 0;
  return g;
}

Sizes measure(const int64_t* off, int64_t nseg) {
  Sizes s;
  if (nseg <= 0) return s;
  s.base = off[0];
  s.keys = off[nseg] - off[0];
  s.chunk = chunk_for(s.keys);
  s.uniform = off[0] == 0 && s.keys > 0;
  long long cut_keys = 0, cut_buckets = 0;  // of the segments that are cut at all
  Seg g{};  // the last segment's, which the next usually equals
  for (int64_t i = 0; i < nseg; ++i) {
    const long long len = off[i + 1] - off[i];
    if (len != off[1] - off[0]) s.uniform = false;
    if (len <= 0) continue;
    ++s.nseg;
    s.longest = std::max(s.longest, len);
    if (len != g.len) g = describe(0, len, s.chunk);
    s.l1.rows += g.rows;
    s.l1.buckets += g.k;
    if (g.k > 1) {
      s.l1.cols += ceil_div(g.k, kCol);
      s.l1.counts += (long long)g.rows * g.k;
      cut_keys += len;
      cut_buckets += g.k;
    }
  }
  s.l1.segs = s.nseg;
  s.small = s.longest <= Large::kCap;
  s.two_levels = s.longest > kOneLevel;
  if (s.two_levels) {
    // Only a bucket of more keys than one workgroup sorts is cut again, and
    // there are few of them: uncut segments and usual buckets have no rows.
    // (One segment of 3 10^6 keys beside 10^6 of 10: 1100 rows and 0.28 GB of
    // scratch, where a row for every segment made 10^6 and 3.2 GB.)
    const long long again = std::min(cut_buckets, cut_keys / (Large::kCap + 1));
    s.l2.segs = s.l1.buckets;
    s.l2.rows = cut_keys / ((long long)s.chunk * kTile) + again;
    s.l2.buckets = cut_keys / kAim + s.l2.segs;
    s.l2.cols = (cut_keys / kAim + again) / kCol + again;
    s.l2.counts = s.l2.rows * buckets_for(s.longest, true);
  }
  return s;
}

// Hands out the scratch in 256-byte pieces.
struct Arena {
  char* base;
  size_t used = 0;
  template <typename T>
  T* take(long long n) {
    T* p = base ? reinterpret_cast<T*>(base + used) : nullptr;
    used += align256(size_t(n) * sizeof(T));
    return p;
  }
};

struct Layout {
  u64* alt;
  Seg *segs1, *segs2;
  Header* bound;
  Level level[2];
  size_t total;
};

Layout lay_out(const Sizes& s, void* scratch) {
  Arena a{reinterpret_cast<char*>(scratch)};
  Layout o{};
  o.alt = a.take<u64>(s.keys);
  unsigned short* ids = a.take<unsigned short>(s.keys);
  Header* headers = a.take<Header>(2);  // overfull buckets; bounds of the second level
  o.bound = headers + 1;
  int* over = a.take<int>(std::max(s.l1.buckets, s.l2.buckets));
  o.segs1 = a.take<Seg>(s.nseg);
  o.segs2 = a.take<Seg>(s.l2.segs);
  for (int i = 0; i < 2; ++i) {
    const LevelSize& z = i ? s.l2 : s.l1;
    Level& l = o.level[i];
    l.chunk = s.chunk;
    l.row_seg = a.take<int>(z.rows);
    l.col_seg = a.take<int>(z.cols);
    l.bucket_seg = a.take<int>(z.buckets);
    l.dup = a.take<int>(z.segs);
    l.splitters = a.take<u64>(z.buckets);
    l.counts = a.take<unsigned>(z.counts);
    l.totals = a.take<unsigned>(z.buckets);
    l.starts = a.take<unsigned>(z.buckets);
    l.ids = ids;
    l.header = headers;
    l.over = over;
  }
  o.total = a.used;
  return o;
}

int partition(u64* x, u64* alt, const Level& l, const LevelSize& z, hipStream_t st) {
  const bool gathered = l.nseg <= kGatherSegs;
  if (gathered) gather_kernel<<<dim3(unsigned(l.nseg * kGather)), dim3(256), 0, st>>>(x, alt, l);
  sample_kernel<<<dim3(unsigned(l.nseg)), dim3(1 << kTB), 0, st>>>(x, alt, l, gathered);
  if (z.rows > 0) {
    hist_kernel<<<dim3(unsigned(z.rows)), dim3(kBS), 0, st>>>(x, alt, l);
    colscan_kernel<<<dim3(unsigned(z.cols)), dim3(kCol * kWalkers), 0, st>>>(l);
    scatter_kernel<<<dim3(unsigned(z.rows)), dim3(kBS), 0, st>>>(x, alt, l);
  }
  return launch_status();
}

}  // namespace

extern "C" {

size_t rpx_sort_segmented_scratch_bytes(const int64_t* offsets_host, int64_t nseg) {
  if (!offsets_host || nseg < 0) return 0;
  const Sizes s = measure(offsets_host, nseg);
  return s.keys > 0 ? lay_out(s, nullptr).total : 0;
}

int rpx_sort_segmented_f64(double* x, const int64_t* offsets_host, int64_t nseg, void* scratch, size_t scratch_bytes,
                           void* stream) {
  if (!offsets_host || nseg < 0) return RPX_ERR_INVALID_ARGUMENT;
  for (int64_t i = 0; i < nseg; ++i) {
    const long long len = offsets_host[i + 1] - offsets_host[i];
    if (offsets_host[i] < 0 || len < 0 || len > INT32_MAX) return RPX_ERR_INVALID_ARGUMENT;
  }
  const Sizes s = measure(offsets_host, nseg);
  if (s.keys == 0) return RPX_SUCCESS;
  if (!x || !scratch) return RPX_ERR_INVALID_ARGUMENT;
  Layout o = lay_out(s, scratch);
  if (scratch_bytes < o.total) return RPX_ERR_SCRATCH_TOO_SMALL;
  if (s.nseg > INT32_MAX || s.l1.buckets > INT32_MAX || s.l2.buckets > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  hipStream_t st = as_stream(stream);
  // x and the scratch copies are indexed alike, from the first segment's key.
  u64* xs = reinterpret_cast<u64*>(x) + s.base;

  Level* l = &o.level[0];
  l->nseg = int(s.nseg);
  if (s.uniform) {
    l->one = describe(0, s.longest, s.chunk);
  } else {
    std::vector<Seg> segs;
    segs.reserve(size_t(s.nseg));
    Seg next{};
    for (int64_t i = 0; i < nseg; ++i) {
      const long long len = offsets_host[i + 1] - offsets_host[i];
      if (len == 0) continue;
      Seg g = describe(offsets_host[i] - s.base, len, s.chunk);
      g.first_row = next.first_row;
      g.first_bucket = next.first_bucket;
      g.first_col = next.first_col;
      g.count_base = next.count_base;
      next.first_row += g.rows;
      next.first_bucket += g.k;
      next.first_col += g.k > 1 ? int(ceil_div(g.k, kCol)) : 0;
      next.count_base += (long long)g.rows * g.k;
      segs.push_back(g);
    }
    const HostChunk table{o.segs1, segs.data(), segs.size() * sizeof(Seg)};
    if (const int rc = upload_async(&table, 1, st); rc != RPX_SUCCESS) return rc;
    l->segs = o.segs1;
  }
  LevelSize z = s.l1;
  if (s.small) {
    l->bucket_seg = nullptr;
  } else {
    if (const int rc = partition(xs, o.alt, *l, z, st); rc != RPX_SUCCESS) return rc;
  }
  if (s.two_levels) {
    Level* l2 = &o.level[1];
    second_level_kernel<<<dim3(1), dim3(1024), 0, st>>>(*l, int(s.l1.buckets), o.segs2, o.bound, s.chunk);
    l2->segs = o.segs2;
    l2->nseg = int(s.l2.segs);
    l2->bound = o.bound;
    l = l2;
    z = s.l2;
    if (const int rc = partition(xs, o.alt, *l, z, st); rc != RPX_SUCCESS) return rc;
  }
  if (s.longest <= Small::kCap)
    bucket_kernel<8><<<dim3(unsigned(z.buckets)), dim3(1 << 8), 0, st>>>(xs, o.alt, *l);
  else
    bucket_kernel<kTB><<<dim3(unsigned(z.buckets)), dim3(1 << kTB), 0, st>>>(xs, o.alt, *l);
  if (!s.small) {
    const unsigned grid = unsigned(z.buckets < 256 ? z.buckets : 256);
    overfull_kernel<<<dim3(grid), dim3(1 << kTB), 0, st>>>(xs, o.alt, *l);
  }
  return launch_status();
}

}  // extern "C"
