// SCAN: exclusive FP64 prefix sum in one pass with decoupled look-back (and
// the inclusive form as an extra output).
//
// Reference: src/algorithm/SCAN.hpp:27-32 (y[i] = s; s += x[i]),
// SCAN-Seq.cpp:31-45, SCAN-OMP.cpp:33-90, SCAN-Hip.cpp:39-326 and the
// suite's grid scan src/common/HipGridScan.hpp:34-197, which memsets its
// ready flags every rep and spins on predecessors indexed by blockIdx.x.
//
// MI355X design:
//  * a tile is 256 or 512 work-items x IPT doubles (IPT 16, 32 or 64: 32-256 KiB).
//    Each wavefront owns a contiguous part of the tile and reads it as
//    IPT/2 rows of 1 KiB (one 16-byte load per lane per row); it scans the
//    rows in order in registers -- lane pair sum, a 64-lane scan on DPP row
//    shifts and row broadcasts, and a running row carry -- so no LDS buffer
//    limits residency, and the result leaves through the same 16-byte row
//    stores.  Row loads and stores are nontemporal unless RPX_TUNE_CACHED is
//    set.  Larger tiles mean fewer look-back hops: 2^28 doubles scan at 4.2,
//    5.1 and 6.0 TB/s with IPT 16, 32 and 64 on MI355X (4.0, 4.9 and 5.5
//    TB/s with the 64-lane scan on ds_bpermute shuffles);
//  * the tile id is the workgroup id: each XCD dispatches its workgroups in
//    id order, so the lowest unfinished tile is always resident and the
//    look-back always makes progress.  (A ticket counter taken with one
//    atomic per tile serialises on its single address -- measured 5.5 ms
//    against 0.8 ms for 2^28 doubles on MI355X.)
//  * the look-back is done by the whole workgroup where there are few tiles
//    and by one wavefront where there are many; a tile's words carry a tag
//    (header epoch + 1) so the scratch needs no clearing between calls.  The
//    last tile advances the epoch after its look-back: by then every tile has
//    published, so every tile has read the epoch;
//  * every spin is bounded; a wait that expires records RPX_ERR_WAIT_EXPIRED
//    in the scratch header and the kernel still runs to completion.
#include "rpx_common.hpp"
#include "scan_words.hpp"

#include <vector>

using namespace rpx;

namespace {

typedef double v2d __attribute__((ext_vector_type(2)));

struct ScanHeader {
  unsigned reserved0;
  unsigned reserved1;
  unsigned long long epoch;
  unsigned error;
};
constexpr size_t kHeaderBytes = 256;
constexpr int kBS = 256;
constexpr int kDefaultIPT = 64;
constexpr int kMinTile = kBS * 16;  // scratch is sized for the smallest tile
constexpr unsigned kSpinLimit = 1u << 22;
constexpr int64_t kWideTiles = 512;  // up to here the whole workgroup looks back

// A tile's look-back state is three 64-bit words.  All move through
// agent-scope atomic loads and stores, which gfx950 performs coherently across
// the XCDs' L2s (sc1), and carry a 42-bit tag (epoch and status) in their top
// bits.
//
// Many tiles: word 0 is a flag, the tag alone, words 1 and 2 the aggregate and
// the inclusive prefix.  Publishing a value before its flag needs only the
// value store to have completed (s_waitcnt vmcnt(0)), not the L2 write-back
// of an agent-scope release fence, which would also flush every dirty output
// line of the XCD; a reader asks for the value once it has the flag.  The
// values are stored complemented: no sum then looks like a tag.
//
// Few tiles (WIDE): each word is the tag over 22 or 21 bits of the value, so
// the writer waits for nothing and a reader takes all three in one round trip
// and retries until their tags agree.  1M doubles as 245 tiles: 8.6 us with
// flags, 5.8 us so and with the whole workgroup looking back.  At 2^28 this
// costs more traffic than it saves waiting: 0.77 against 0.71 ms.
struct TileWords {
  unsigned long long *w0, *w1, *w2;  // [tile]
};
constexpr int kLowBits = 21;  // of words 1 and 2; word 0 holds the top 22
constexpr unsigned long long kLowMask = (1ull << kLowBits) - 1;

__device__ __forceinline__ void store_word(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long load_word(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long bits(double v) {
  return static_cast<unsigned long long>(__double_as_longlong(v));
}
__device__ __forceinline__ double value(unsigned long long b) { return __longlong_as_double(static_cast<long long>(b)); }

template <bool WIDE>
__device__ __forceinline__ void publish(const TileWords& w, int64_t t, unsigned long long epoch, unsigned status,
                                        double v) {
  const unsigned long long b = bits(v), tag = tile_tag(epoch, status);
  if constexpr (WIDE) {
    store_word(&w.w0[t], tag | b >> (2 * kLowBits));
    store_word(&w.w1[t], tag | (b >> kLowBits & kLowMask));
    store_word(&w.w2[t], tag | (b & kLowMask));
  } else {
    store_word(status == 2 ? &w.w2[t] : &w.w1[t], ~b);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // compiler ordering
    __builtin_amdgcn_s_waitcnt(0x0F70);                      // vmcnt(0): value store complete
    store_word(&w.w0[t], tag);
  }
}
// The status of tile k in this epoch, 0 if it has none yet (or, WIDE, is being
// rewritten); WIDE: *v is its value.
template <bool WIDE>
__device__ __forceinline__ unsigned look(const TileWords& w, int64_t k, unsigned long long epoch, double* v) {
  const unsigned long long a = load_word(&w.w0[k]);
  if constexpr (WIDE) {
    const unsigned long long b = load_word(&w.w1[k]), c = load_word(&w.w2[k]), tag = a >> 22;
    if (b >> 22 != tag || c >> 22 != tag) return 0;
    *v = value((a & 0x3FFFFFull) << (2 * kLowBits) | (b & kLowMask) << kLowBits | (c & kLowMask));
  }
  return tile_status(a, epoch);
}

// Wavefront scans on DPP lane moves (VALU only, no LDS round trips).  A
// 64-bit value moves as two 32-bit halves; lanes whose source is outside
// the pattern, or in a row the mask leaves out, receive 0.
template <int CTRL, int ROW_MASK, bool ZERO_FILL>
__device__ __forceinline__ double dpp_move(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(b), CTRL, ROW_MASK, 0xF, ZERO_FILL);
  const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), CTRL, ROW_MASK, 0xF, ZERO_FILL);
  return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(unsigned(hi)) << 32) |
                                                     unsigned(lo)));
}

// Inclusive scan over the 64 lanes: shifts by 1, 2, 4 and 8 within each row
// of 16 lanes, then lane 15's row total into rows 1 and 3 (row_bcast:15)
// and lane 31's half total into rows 2 and 3 (row_bcast:31).
__device__ __forceinline__ double wave_inclusive_scan_dpp(double v) {
  v += dpp_move<0x111, 0xF, false>(v);  // row_shr:1
  v += dpp_move<0x112, 0xF, false>(v);  // row_shr:2
  v += dpp_move<0x114, 0xF, false>(v);  // row_shr:4
  v += dpp_move<0x118, 0xF, false>(v);  // row_shr:8
  v += dpp_move<0x142, 0xA, false>(v);  // row_bcast:15
  v += dpp_move<0x143, 0xC, false>(v);  // row_bcast:31
  return v;
}

// Lane l receives lane l-1's value, lane 0 receives 0 (wave_shr:1).
__device__ __forceinline__ double wave_shift_up_dpp(double v) { return dpp_move<0x138, 0xF, true>(v); }
// Lane l receives lane l+1's value, lane 63 receives 0 (wave_shl:1).
__device__ __forceinline__ double wave_shift_down_dpp(double v) { return dpp_move<0x130, 0xF, true>(v); }

// Lane L's value, wavefront-uniform.
template <int L>
__device__ __forceinline__ double lane_value(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane(int(b), L);
  const int hi = __builtin_amdgcn_readlane(int(b >> 32), L);
  return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(unsigned(hi)) << 32) |
                                                     unsigned(lo)));
}
__device__ __forceinline__ double last_lane(double v) { return lane_value<kWave - 1>(v); }

// One wavefront's look at the 64 tiles top, top - 1, ... (tiles before `first`
// count as an inclusive prefix of zero): the sum of their values back to and
// with the nearest inclusive one, *done if there is one.
template <bool WIDE>
__device__ __forceinline__ double look_window(const TileWords& words, int64_t top, int64_t first,
                                              unsigned long long epoch, int lane, bool* done, bool* expired) {
  const int64_t k = top - lane;
  double val = 0.0;
  unsigned status = 2;
  if (k >= first) {
    unsigned spins = 0;
    while ((status = look<WIDE>(words, k, epoch, &val)) == 0) {
      if (++spins > kSpinLimit) {
        *expired = true;
        status = 2;
        val = 0.0;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // value loads stay after the flag tests
  const unsigned long long inc = __ballot(status == 2);
  const int last = inc ? __ffsll(static_cast<long long>(inc)) - 1 : kWave;
  *done = inc != 0;
  if (!WIDE && k >= first && !*expired) {
    if (lane < last) val = value(~load_word(&words.w1[k]));
    else if (lane == last) val = value(~load_word(&words.w2[k]));
  }
  return wave_sum(lane <= last ? val : 0.0);
}

// Segment tables of a segmented scan: segment s covers [off[s], off[s+1])
// and owns the global tiles [tile0[s], tile0[s+1]); tile t belongs to
// segment tile_seg[t].  A segment's tiles start at even elements (the
// segment's start rounded down to even, then whole tiles), so every tile
// after its first reads and writes 16-byte rows; the first tile skips the
// element before an odd start.
struct SegTables {
  const uint64_t* off;       // table_entry
  const uint64_t* tile0;     // table_entry
  const uint32_t* tile_seg;  // segment_entry
};

// SEG = false: one array of n elements, tile t covers [t*T, t*T + T), words
// carry the epoch read from the header.  SEG = true: tiles come from the
// segment tables, the look-back stops at the segment's first tile, and the
// words were cleared before the launch (epoch 0, no epoch advance).
template <int BS, int ROWS, bool NT, bool SEG, bool INCL, bool WIDE>  // 16-byte rows per lane: 128*ROWS doubles a wave
__global__ __launch_bounds__(BS) void scan_kernel(const double* x, double* y, int64_t n, int64_t ntiles,
                                                   ScanHeader* __restrict__ hdr, TileWords words, int vec,
                                                   SegTables seg) {
  constexpr int kRowLen = 2 * kWave;            // doubles per wavefront row
  constexpr int kChunk = kRowLen * ROWS;        // doubles per wavefront
  constexpr int kTileN = kChunk * (BS / kWave);
  __shared__ double wave_tot[BS / kWave];
  __shared__ unsigned long long s_epoch;
  __shared__ double look_sum[2][BS / kWave];
  __shared__ int look_done[2][BS / kWave];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  if (!SEG && tid == 0) s_epoch = __hip_atomic_load(&hdr->epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  const int64_t t = blockIdx.x;
  // The tile spans [tal, tal + kTileN) from an even tal and owns the
  // elements [lo, tend) of it; first is its segment's first tile.
  int64_t tal, lo, tend, first;
  if (SEG) {
    const int sg = segment_value(seg.tile_seg[t]);
    first = table_value(seg.tile0[sg]);
    const int64_t sbeg = table_value(seg.off[sg]), send = table_value(seg.off[sg + 1]);
    tal = (sbeg & ~int64_t(1)) + (t - first) * kTileN;
    lo = sbeg > tal ? sbeg : tal;
    tend = (tal + kTileN < send) ? tal + kTileN : send;
  } else {
    first = 0;
    tal = lo = t * kTileN;
    tend = (tal + kTileN < n) ? tal + kTileN : n;
  }
  const int64_t base = tal + int64_t(wave) * kChunk + 2 * lane;
  // x and y are 16-byte aligned (vec) and tal is even, so the rows are too.
  const bool full = vec && lo == tal && tend - tal == kTileN;
  n = tend;  // bounds of the partial-tile paths below

  // Each wavefront owns a contiguous chunk, read as ROWS coalesced 1 KiB rows.
  v2d v[ROWS];
  if (full) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const v2d* p = reinterpret_cast<const v2d*>(x + base + r * kRowLen);
      v[r] = NT ? __builtin_nontemporal_load(p) : *p;
    }
  } else {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int64_t i0 = base + r * kRowLen;
      v[r].x = (i0 >= lo && i0 < n) ? x[i0] : 0.0;
      v[r].y = (i0 + 1 >= lo && i0 + 1 < n) ? x[i0 + 1] : 0.0;
    }
  }

  // Exclusive scan inside the wavefront, row by row: lane pair sums, a
  // 64-lane scan on DPP moves, and a running carry of the row totals.  The
  // pair sum replaces the pair's second element, so each row keeps two
  // values; the inclusive form (INCL) is built from these exclusive values
  // when it is stored.
  double carry = 0.0;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const double p = v[r].x + v[r].y;
    const double inc = wave_inclusive_scan_dpp(p);
    const double exc = wave_shift_up_dpp(inc);
    const double row_total = last_lane(inc);
    const double e0 = carry + exc;
    v[r] = v2d{e0, e0 + v[r].x};
    carry += row_total;
  }
  if (lane == 0) wave_tot[wave] = carry;
  __syncthreads();
  // Epoch: 0 for the segmented form (its words are cleared before every
  // launch), the header's + 1 for the single-array form, so a single-array scan
  // never accepts a word or table entry a segmented call left in a shared
  // scratch.
  const unsigned long long E = SEG ? 0ull : (s_epoch + 1) & 0xFFFFFFFFFFull;
  double wave_off = 0.0, tile_agg = 0.0;
#pragma unroll
  for (int w = 0; w < BS / kWave; ++w) {
    const double wt = wave_tot[w];
    if (w < wave) wave_off += wt;
    tile_agg += wt;
  }
  if (tid == 0) publish<WIDE>(words, t, E, t == first ? 2 : 1, tile_agg);

  // Look back.  Few tiles all publish at about the same time, so there the
  // whole workgroup looks, BS predecessors per round; many tiles find an
  // inclusive prefix close by, and wavefront 0 looks alone (looking BS back at
  // 2^28 doubles waits for tiles it does not need, and took 1.00 ms).
  double prefix = 0.0;
  if (WIDE && t != first) {
    bool expired = false;
    int64_t top = t - 1;
    for (int round = 0;; round ^= 1, top -= BS) {
      bool done;
      const double sum = look_window<true>(words, top - int64_t(wave) * kWave, first, E, lane, &done, &expired);
      if (lane == 0) {
        look_sum[round][wave] = sum;
        look_done[round][wave] = done;
      }
      __syncthreads();
      done = false;
#pragma unroll
      for (int w = 0; w < BS / kWave; ++w) {
        if (!done) prefix += look_sum[round][w];
        done |= look_done[round][w] != 0;
      }
      if (done) break;
    }
    if (tid == 0) publish<WIDE>(words, t, E, 2, prefix + tile_agg);
    if (expired) atomicOr(&hdr->error, 1u);
  } else if (t != first) {
    if (wave == 0) {
      bool expired = false, done = false;
      for (int64_t top = t - 1; !done; top -= kWave) prefix += look_window<false>(words, top, first, E, lane, &done, &expired);
      if (lane == 0) {
        publish<WIDE>(words, t, E, 2, prefix + tile_agg);
        look_sum[0][0] = prefix;
      }
      if (expired) atomicOr(&hdr->error, 1u);
    }
    __syncthreads();
    prefix = look_sum[0][0];
  }
  // Every tile has read the epoch once the last tile's look-back is done.
  if (!SEG && tid == 0 && t == ntiles - 1) atomicAdd(&hdr->epoch, 1ull);

  const double off = prefix + wave_off;
  // The inclusive value of an element is the exclusive value of the element
  // after it: for lane l's pair, its own second value and lane l+1's first
  // (for lane 63 the next row's first, after the last row the wavefront's
  // total).  Element n-1 of a partial tile takes the same rule, since the
  // padding beyond n is zero.
  if constexpr (INCL) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const double next = (r + 1 < ROWS) ? lane_value<0>(v[r + 1].x) : carry;
      const double shifted = wave_shift_down_dpp(v[r].x);
      v[r] = v2d{v[r].y, lane == kWave - 1 ? next : shifted};
    }
  }
  if (full) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      v2d* p = reinterpret_cast<v2d*>(y + base + r * kRowLen);
      const v2d o = v2d{off + v[r].x, off + v[r].y};
      if (NT) __builtin_nontemporal_store(o, p);
      else *p = o;
    }
  } else {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int64_t i0 = base + r * kRowLen;
      if (i0 >= lo && i0 < n) y[i0] = off + v[r].x;
      if (i0 + 1 >= lo && i0 + 1 < n) y[i0 + 1] = off + v[r].y;
    }
  }
}

__global__ void zero_kernel(unsigned* p, int64_t nwords) {
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < nwords; i += stride) p[i] = 0u;
}

// Before a segmented scan: clears the tiles' words and fills tile_seg from tile0
// (the last segment whose first tile is <= t owns tile t; empty segments
// share their first tile with the next segment and so are never chosen).
__global__ __launch_bounds__(256) void seg_prep_kernel(unsigned* __restrict__ words, int64_t nwords,
                                                       const uint64_t* __restrict__ tile0, int nseg,
                                                       uint32_t* __restrict__ tile_seg, int64_t ntiles) {
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  const int64_t entries = ntiles + (ntiles & 1);  // whole 64 bits
  const int64_t end = nwords > entries ? nwords : entries;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < end; i += stride) {
    if (i < nwords) words[i] = 0u;
    if (i < entries) {
      int a = 0, b = nseg - 1;
      while (a < b) {
        const int mid = (a + b + 1) >> 1;
        if (table_value(tile0[mid]) <= i) a = mid;
        else b = mid - 1;
      }
      tile_seg[i] = segment_entry(a);
    }
  }
}

inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

struct Layout {
  size_t words_off[3], total;
};
Layout layout_for(int64_t ntiles) {
  Layout l;
  l.total = kHeaderBytes;
  for (size_t& off : l.words_off) {
    off = l.total;
    l.total += align256(size_t(ntiles) * 8);
  }
  return l;
}
TileWords words_in(char* base, const Layout& l) {
  auto at = [&](int i) { return reinterpret_cast<unsigned long long*>(base + l.words_off[i]); };
  return {at(0), at(1), at(2)};
}

template <int ROWS, bool SEG, int BS = kBS, bool INCL = false>
void launch_rows(bool nt, unsigned grid, const double* x, double* y, int64_t n, int64_t ntiles, ScanHeader* hdr,
                 TileWords words, int vec, SegTables seg, hipStream_t s) {
  const bool wide = !SEG && ROWS <= 8 && ntiles <= kWideTiles;
  auto go = [&](auto kernel) { kernel<<<dim3(grid), dim3(BS), 0, s>>>(x, y, n, ntiles, hdr, words, vec, seg); };
  if constexpr (!SEG && ROWS <= 8) {
    if (wide) return nt ? go(scan_kernel<BS, ROWS, true, SEG, INCL, true>) : go(scan_kernel<BS, ROWS, false, SEG, INCL, true>);
  }
  if (nt) go(scan_kernel<BS, ROWS, true, SEG, INCL, false>);
  else go(scan_kernel<BS, ROWS, false, SEG, INCL, false>);
}

// Default tile: 64 doubles for each of 256 work-items, and smaller ones where
// that would leave most CUs without a tile (and the scratch has their words):
// 1M doubles take 11.3 us as 62 tiles of 16384 and 8.6 us as 245 of 4096; at
// 4M tiles of 8192 (512 work-items) are the fastest, 15.3 us against 16.0 and
// 18.4.
constexpr int64_t kSmallScan = int64_t(1) << 20, kMediumScan = int64_t(1) << 22;
struct ScanShape {
  int bs, ipt;
};
ScanShape scan_shape(int64_t n, const rpx_tuning* tune, size_t scratch_bytes) {
  const int bs = tune_or(tune, &rpx_tuning::block_size, 0), ipt = tune_or(tune, &rpx_tuning::items_per_thread, 0);
  if (bs == 0 && ipt == 0 && n <= kMediumScan) {
    const ScanShape d{n <= kSmallScan ? 256 : 512, 16};
    if (layout_for(ceil_div(n, int64_t(d.bs) * d.ipt)).total <= scratch_bytes) return d;
  }
  return {bs ? bs : kBS, ipt ? ipt : kDefaultIPT};
}

template <bool INCL>
int scan_one(const double* x, double* y, int64_t n, int ipt, int bs, bool nt, void* scratch, size_t scratch_bytes,
             hipStream_t s) {
  if (n == 0) return RPX_SUCCESS;
  if (ipt != 16 && ipt != 32 && ipt != 64) return RPX_ERR_INVALID_ARGUMENT;
  if (bs != 256 && bs != 512) return RPX_ERR_INVALID_ARGUMENT;
  const int64_t ntiles = ceil_div(n, int64_t(bs) * ipt);
  if (ntiles > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  const Layout l = layout_for(ntiles);
  if (scratch_bytes < l.total) return RPX_ERR_SCRATCH_TOO_SMALL;
  char* base = reinterpret_cast<char*>(scratch);
  auto* hdr = reinterpret_cast<ScanHeader*>(base);
  const TileWords words = words_in(base, l);
  const int vec = aligned16(x) && aligned16(y);
  const unsigned grid = unsigned(ntiles);
  const SegTables none{nullptr, nullptr, nullptr};
  if (bs == 512) {
    if (ipt == 16) launch_rows<8, false, 512, INCL>(nt, grid, x, y, n, ntiles, hdr, words, vec, none, s);
    else if (ipt == 32)
      launch_rows<16, false, 512, INCL>(nt, grid, x, y, n, ntiles, hdr, words, vec, none, s);
    else launch_rows<32, false, 512, INCL>(nt, grid, x, y, n, ntiles, hdr, words, vec, none, s);
  } else {
    if (ipt == 16) launch_rows<8, false, kBS, INCL>(nt, grid, x, y, n, ntiles, hdr, words, vec, none, s);
    else if (ipt == 32)
      launch_rows<16, false, kBS, INCL>(nt, grid, x, y, n, ntiles, hdr, words, vec, none, s);
    else launch_rows<32, false, kBS, INCL>(nt, grid, x, y, n, ntiles, hdr, words, vec, none, s);
  }
  return launch_status();
}

// Segmented scan: every tile of every segment in one launch (tiles of
// 256 x 64 doubles from the segment's even-rounded start; a segment's first
// and last tiles may be partial).  Scratch: the single-array layout for the
// total tile count, then off[nseg+1] and tile0[nseg+1] (one upload), then
// tile_seg[ntiles] (filled on the device).
constexpr int64_t kSegTile = int64_t(kBS) * kDefaultIPT;

inline int64_t seg_tiles(int64_t sbeg, int64_t send) {
  return send > sbeg ? ceil_div(send - (sbeg & ~int64_t(1)), kSegTile) : 0;
}

struct SegLayout {
  Layout l;
  int64_t ntiles;
  size_t tab_off, tile_seg_off, total;
};
SegLayout seg_layout(const int64_t* offsets_host, int64_t nseg) {
  SegLayout g;
  g.ntiles = 0;
  for (int64_t s = 0; s < nseg; ++s) g.ntiles += seg_tiles(offsets_host[s], offsets_host[s + 1]);
  g.l = layout_for(g.ntiles > 0 ? g.ntiles : 1);
  g.tab_off = g.l.total;
  g.tile_seg_off = g.tab_off + align256(size_t(2 * (nseg + 1)) * sizeof(int64_t));
  g.total = g.tile_seg_off + align256(size_t(g.ntiles) * sizeof(uint32_t));
  return g;
}

}  // namespace

extern "C" {

size_t rpx_scan_scratch_bytes(int64_t n, const rpx_tuning* /*tune*/) {
  if (n < 0) return 0;
  return layout_for(ceil_div(n > 0 ? n : 1, kMinTile)).total;
}

int rpx_scan_exclusive_f64(const double* x, double* y, int64_t n, void* scratch, size_t scratch_bytes,
                           const rpx_tuning* tune, void* stream) {
  if (n < 0 || (n > 0 && (!x || !y || !scratch))) return RPX_ERR_INVALID_ARGUMENT;
  const ScanShape d = scan_shape(n, tune, scratch_bytes);
  const bool nt = (tune_flags(tune) & RPX_TUNE_CACHED) == 0;
  return scan_one<false>(x, y, n, d.ipt, d.bs, nt, scratch, scratch_bytes, as_stream(stream));
}

int rpx_scan_inclusive_f64(const double* x, double* y, int64_t n, void* scratch, size_t scratch_bytes,
                           const rpx_tuning* tune, void* stream) {
  if (n < 0 || (n > 0 && (!x || !y || !scratch))) return RPX_ERR_INVALID_ARGUMENT;
  const ScanShape d = scan_shape(n, tune, scratch_bytes);
  const bool nt = (tune_flags(tune) & RPX_TUNE_CACHED) == 0;
  return scan_one<true>(x, y, n, d.ipt, d.bs, nt, scratch, scratch_bytes, as_stream(stream));
}

size_t rpx_scan_segmented_scratch_bytes(const int64_t* offsets_host, int64_t nseg) {
  if (!offsets_host || nseg < 0 || nseg > INT32_MAX) return 0;
  for (int64_t s = 0; s < nseg; ++s)
    if (offsets_host[s + 1] < offsets_host[s]) return 0;
  return seg_layout(offsets_host, nseg).total;
}

int rpx_scan_exclusive_segmented_f64(const double* x, double* y, const int64_t* offsets_host, int64_t nseg,
                                     void* scratch, size_t scratch_bytes, void* stream) {
  if (!offsets_host || nseg < 0 || nseg > INT32_MAX || !scratch) return RPX_ERR_INVALID_ARGUMENT;
  for (int64_t s = 0; s < nseg; ++s)
    if (offsets_host[s + 1] < offsets_host[s] || offsets_host[s] < 0) return RPX_ERR_INVALID_ARGUMENT;
  if (nseg > 0 && offsets_host[nseg] > 0 && (!x || !y)) return RPX_ERR_INVALID_ARGUMENT;
  const SegLayout g = seg_layout(offsets_host, nseg);
  if (scratch_bytes < g.total) return RPX_ERR_SCRATCH_TOO_SMALL;
  if (g.ntiles == 0) return RPX_SUCCESS;
  if (g.ntiles > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  hipStream_t st = as_stream(stream);
  char* base = reinterpret_cast<char*>(scratch);
  // Tables: the offsets, then each segment's first tile (one copy).
  std::vector<uint64_t> tab(size_t(2 * (nseg + 1)));
  int64_t t = 0;
  for (int64_t s = 0; s <= nseg; ++s) {
    tab[size_t(s)] = table_entry(offsets_host[s]);
    tab[size_t(nseg + 1 + s)] = table_entry(t);
    if (s < nseg) t += seg_tiles(offsets_host[s], offsets_host[s + 1]);
  }
  auto* d_off = reinterpret_cast<uint64_t*>(base + g.tab_off);
  auto* d_tile0 = d_off + (nseg + 1);
  auto* d_tile_seg = reinterpret_cast<uint32_t*>(base + g.tile_seg_off);
  const HostChunk table{d_off, tab.data(), tab.size() * sizeof(uint64_t)};
  if (const int rc = upload_async(&table, 1, st); rc != RPX_SUCCESS) return rc;
  // The tiles' words start at zero for every call (no epochs across segments).
  char* const tiles = base + g.l.words_off[0];
  const int64_t words = int64_t(g.l.total - g.l.words_off[0]) / 4;
  const int64_t work = words > g.ntiles ? words : g.ntiles;
  seg_prep_kernel<<<dim3(unsigned(ceil_div(work, 256) < 4096 ? ceil_div(work, 256) : 4096)), dim3(256), 0, st>>>(
      reinterpret_cast<unsigned*>(tiles), words, d_tile0, int(nseg), d_tile_seg, g.ntiles);
  if (const int rc = launch_status(); rc != RPX_SUCCESS) return rc;
  const SegTables seg{d_off, d_tile0, d_tile_seg};
  const int vec = aligned16(x) && aligned16(y);
  launch_rows<32, true>(true, unsigned(g.ntiles), x, y, offsets_host[nseg], g.ntiles,
                        reinterpret_cast<ScanHeader*>(base), words_in(base, g.l), vec, seg, st);
  return launch_status();
}

// Zeroes a scan scratch buffer; required once before its first use.
int rpx_scan_scratch_init(void* scratch, size_t scratch_bytes, void* stream) {
  if (!scratch || scratch_bytes < kHeaderBytes) return RPX_ERR_INVALID_ARGUMENT;
  const int64_t words = int64_t(scratch_bytes / 4);
  int64_t g = ceil_div(words, 256);
  if (g > 4096) g = 4096;
  zero_kernel<<<dim3(unsigned(g)), dim3(256), 0, as_stream(stream)>>>(reinterpret_cast<unsigned*>(scratch), words);
  return launch_status();
}

// Reads the scratch header's error word (synchronous).
int rpx_scan_scratch_status(const void* scratch) {
  if (!scratch) return RPX_ERR_INVALID_ARGUMENT;
  ScanHeader h;
  RPX_TRY(hipMemcpy(&h, scratch, sizeof(h), hipMemcpyDeviceToHost));
  return h.error ? RPX_ERR_WAIT_EXPIRED : RPX_SUCCESS;
}

}  // extern "C"
