// Mixed-precision GEMM with FP64 accuracy from int8 matrix cores.
//
// Same result semantics as the suite's GEMM (src/polybench/POLYBENCH_GEMM.hpp
// :12-50: C = alpha*A*B, beta never reaches C).  The product is emulated
// with the modular integer scheme of Ozaki, Uchino & Imamura ("Ozaki scheme
// II", 2025): one int8 GEMM per modulus instead of one per pair of
// fixed-point slices.
//   * Row i of A is scaled by 2^(b-e_i) and column j of B by 2^(b-f_j),
//     where 2^(e_i-1) <= max_k |A[i][k]| < 2^e_i (likewise f_j), and rounded
//     to integers: |A'|, |B'| <= 2^b.  X = A'B' is an exact integer with
//     |X| <= nk 4^b.
//   * T pairwise coprime moduli m_t <= 256 (the largest such numbers) with
//     M = prod m_t > 2 nk 4^b.  For each t the symmetric residues of A' and
//     B' lie in [-128, 128] (128 only for m_t = 256, where it is stored as
//     the byte -128, the same residue) and one GEMM on
//     v_mfma_i32_16x16x64_i8 gives their product exactly in int32 (nk <=
//     131071); its epilogue keeps d_t = that product modulo m_t, a
//     symmetric residue of X, one byte per output.
//   * Chinese remainder theorem: X = sum_t d_t y_t M/m_t (mod M), y_t =
//     (M/m_t)^-1 mod m_t, so X/M = sum_t d_t y_t/m_t minus the nearest
//     integer, |X/M| < 1/2.  With y_t/m_t = h_t + l_t, h_t a multiple of
//     2^-44, the sum of d_t h_t is kept exactly in FP64 modulo 1 and the sum
//     of d_t l_t (below T 2^-36) is added after the integer part is removed,
//     so X comes out with a relative error of a few 2^-53, plus an absolute
//     error below 2^-84 M, however much it cancels.
//   * C[i][j] = alpha 2^(e_i+f_j-2b) X.
// The only approximation is the rounding of A and B to b bits below their
// row/column maxima: |C - alpha AB|_ij <= |alpha| 2^(e_i+f_j-b) nk (1+2^-b)
// plus FP64 rounding of the result.  b is the largest value with
// 2 nk 4^b < M, at most 46 (so every quotient below is exact, see
// sym_mod); by default T is the smallest count giving b >= 42 (13 moduli,
// b = 44 at nk = 4096), an error below 2^-42 relative to
// |alpha| max_k|A[i][k]| max_k|B[k][j]| nk.
//
// Scratch holds the int8 residues (A: [t][i][k], B: [t][j][k], K
// contiguous, zero-padded to tile multiples), the per-row/column exponents
// and the residue bytes d_t ([t] then the GEMM's accumulator fragments).
#include "rpx_common.hpp"

#include <algorithm>

using namespace rpx;

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kMaxMods = 16;
// The 16 largest pairwise coprime integers not above 256.
constexpr int kMods[kMaxMods] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193};
constexpr int kMinBits = 42;       // automatic modulus count: the smallest T with b >= 42
constexpr int kMaxBits = 46;       // |A'|, |B'| <= 2^46: exact quotients in sym_mod
constexpr int64_t kMaxK = 131071;  // 128 * 128 * nk < 2^31

constexpr int kTM = 256, kTN = 256, kTK = 128;  // block tile, K bytes per stage
constexpr int kChunks = kTK / 16;               // 16-byte chunks per tile row and stage

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }
inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// Per-call constants of the modular scheme, passed by value to the kernels.
struct CrtParams {
  int T, b;
  double inv[kMaxMods];         // fl(1/m_t)
  unsigned minus_m[kMaxMods];   // -m_t modulo 256
  double h[kMaxMods];    // floor(2^44 y_t/m_t) 2^-44, y_t = (M/m_t)^-1 mod m_t
  double l[kMaxMods];    // y_t/m_t - h_t, rounded
  double M_hi, M_lo;     // prod m_t = M_hi + M_lo, M_lo rounded (a 2^-106 relative error)
};

typedef unsigned __int128 u128;

int64_t inverse_mod(int64_t a, int64_t m) {
  int64_t t = 0, nt = 1, r = m, nr = a % m;
  while (nr != 0) {
    const int64_t q = r / nr;
    int64_t tmp = t - q * nt; t = nt; nt = tmp;
    tmp = r - q * nr; r = nr; nr = tmp;
  }
  return t < 0 ? t + m : t;
}

// Largest b <= kMaxBits with 2 nk 4^b < M, or -1.
int bits_for(int64_t nk, int T) {
  u128 M = 1;
  for (int t = 0; t < T; ++t) M *= u128(kMods[t]);
  const u128 k = u128(nk > 0 ? nk : 1);
  for (int b = kMaxBits; b >= 0; --b)
    if (2 * k * (u128(1) << (2 * b)) < M) return b;
  return -1;
}

int moduli_for(int64_t nk, int nmoduli) {
  if (nmoduli > 0) return nmoduli;
  for (int T = 1; T <= kMaxMods; ++T)
    if (bits_for(nk, T) >= kMinBits) return T;
  return kMaxMods;
}

bool crt_setup(int64_t nk, int nmoduli, CrtParams* p) {
  const int T = moduli_for(nk, nmoduli);
  if (T < 1 || T > kMaxMods) return false;
  const int b = bits_for(nk, T);
  if (b < 1) return false;
  p->T = T;
  p->b = b;
  u128 M = 1;
  for (int t = 0; t < T; ++t) M *= u128(kMods[t]);
  // M < 2^126 fits long double's range; hi is an integer, so hiu = hi exactly
  // and M - hi (below 2^73 in magnitude) is exact in 128-bit integers
  // before its rounding to FP64.
  const double hi = double(static_cast<long double>(M));
  const u128 hiu = static_cast<u128>(static_cast<long double>(hi));
  p->M_hi = hi;
  p->M_lo = hiu >= M ? -double(static_cast<long double>(hiu - M)) : double(static_cast<long double>(M - hiu));
  for (int t = 0; t < kMaxMods; ++t) {
    const int64_t m = kMods[t];
    p->minus_m[t] = unsigned(-m) & 0xFFu;
    p->inv[t] = 1.0 / double(m);
    int64_t mt = 1;  // (M / m_t) mod m_t
    for (int s = 0; s < T; ++s)
      if (s != t) mt = mt * kMods[s] % m;
    const uint64_t y = t < T ? uint64_t(inverse_mod(mt, m)) : 0;
    const uint64_t num = y << 44;  // y < 256: below 2^52
    p->h[t] = std::ldexp(double(num / uint64_t(m)), -44);
    p->l[t] = std::ldexp(double(num % uint64_t(m)) / double(m), -44);
  }
  return true;
}

struct MixedLayout {
  int64_t nip, njp, nkp;
  size_t a_off, b_off, ea_off, fb_off, r_off, total;
};
MixedLayout mixed_layout(int64_t ni, int64_t nj, int64_t nk, int T) {
  MixedLayout l;
  l.nip = round_up(ni, kTM);
  l.njp = round_up(nj, kTN);
  l.nkp = round_up(nk > 0 ? nk : 1, 2 * kTK);  // the K loop takes two stages per step
  l.a_off = 0;
  l.b_off = align256(size_t(T) * l.nip * l.nkp);
  l.ea_off = l.b_off + align256(size_t(T) * l.njp * l.nkp);
  l.fb_off = l.ea_off + align256(size_t(l.nip) * 4);
  l.r_off = l.fb_off + align256(size_t(l.njp) * 4);
  l.total = l.r_off + align256(size_t(T) * l.nip * l.njp);  // d_t, one byte per output
  return l;
}

__device__ __forceinline__ int exponent_of(double m) {
  int e = 0;
  if (m != 0.0) frexp(m, &e);
  return e;
}

// Symmetric residue of the integer-valued x modulo m, |x| <= 2^46 (or
// |x| < 2^31), in the low byte of the result; the other bytes are anything.
// x fl(1/m) is within 2^-15 of x/m, and x/m is at least 1/(2m) >= 2^-9 from a
// half-integer unless m = 256 and x = 128 (mod 256).  So the fma, rounded to
// integers by the size of kInteger, has rint(x/m) in its low bits, and the
// residue x - rint(x/m) m lies in [-(m-1)/2, (m-1)/2], or in [-128, 128] for
// m = 256, where the byte kept makes 128 the same residue as -128.  Only its
// low byte is wanted, so the low bytes of x, of the quotient and of -m do:
// one FP64 instruction and one 24-bit multiply-add where the residue as a
// double and its conversion took four FP64 instructions.
constexpr double kInteger = 6755399441055744.0;  // 1.5 * 2^52
__device__ __forceinline__ unsigned low_word(double x) { return unsigned(__double2loint(x + kInteger)); }
__device__ __forceinline__ unsigned sym_mod(double x, unsigned x_low, double inv, unsigned minus_m) {
  return __umul24(unsigned(__double2loint(fma(x, inv, kInteger))), minus_m) + x_low;
}
// The low bytes of four words.
__device__ __forceinline__ unsigned pack4(unsigned a, unsigned b, unsigned c, unsigned d) {
  return __builtin_amdgcn_perm(b, a, 0x0c0c0400u) | __builtin_amdgcn_perm(d, c, 0x04000c0cu);
}

// Row i of A (padded rows too) by one workgroup: row exponent, then the
// residues.  A work-item takes four consecutive k of every 1024, so that a
// wavefront's loads and, per modulus, its stores are whole lines, and up to
// 4096 k stay in registers between the two uses (with 16 consecutive k per
// work-item a wavefront's load touched 64 lines, which had left the L1 before
// the next load wanted them: 4096 rows of 4096 took 83 us, 66
// here with the cheaper residues, 54 for its bytes).
constexpr int kRowPasses = 4, kRowSpan = kRowPasses * 1024;
__device__ __forceinline__ void split_row(const double* __restrict__ A, int64_t i, int64_t ni, int64_t nk, int64_t nkp,
                                          int64_t nip, signed char* __restrict__ As, int* __restrict__ ea,
                                          const CrtParams& P, double* red) {
  const int tid = threadIdx.x;
  const bool live = i < ni;
  const double* row = A + (live ? i * nk : 0);
  double x[4 * kRowPasses];
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int p = 0; p < kRowPasses; ++p) {
      const int64_t k = k0 + 1024 * p + 4 * tid;
      if (live && k + 4 <= nk) {
#pragma unroll
        for (int c = 0; c < 4; ++c) x[4 * p + c] = row[k + c];
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) x[4 * p + c] = live && k + c < nk ? row[k + c] : 0.0;
      }
    }
  };
  double m = 0.0;
  for (int64_t k0 = 0; k0 < nkp; k0 += kRowSpan) {
    load(k0);
#pragma unroll
    for (int u = 0; u < 4 * kRowPasses; ++u) m = fmax(m, fabs(x[u]));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  const int e = exponent_of(m);
  if (tid == 0) ea[i] = e;
  for (int64_t k0 = 0; k0 < nkp; k0 += kRowSpan) {
    if (nkp > kRowSpan) load(k0);
#pragma unroll
    for (int p = 0; p < kRowPasses; ++p) {
      const int64_t k = k0 + 1024 * p + 4 * tid;
      if (k >= nkp) continue;
      double v[4];
      unsigned low[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        v[c] = rint(ldexp(x[4 * p + c], P.b - e));
        low[c] = low_word(v[c]);
      }
      signed char* out = As + i * nkp + k;
      for (int t = 0; t < P.T; ++t, out += nip * nkp) {
        unsigned r[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) r[c] = sym_mod(v[c], low[c], P.inv[t], P.minus_m[t]);
        *reinterpret_cast<unsigned*>(out) = pack4(r[0], r[1], r[2], r[3]);
      }
    }
  }
}

// Maxima of 64 columns of B over the rows [k0, ke), as exponents (INT32_MIN for
// a column of zeros): wavefront w reads rows w, w + 4, ... (each load is 64
// consecutive columns of one row, 16 loads in flight per work-item), and the
// four wavefronts' maxima meet in LDS.
__device__ __forceinline__ void column_exponents(const double* __restrict__ B, int64_t j0, int64_t k0, int64_t ke,
                                                 int64_t nj, int* __restrict__ out, double* red) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t j = j0 + lane;
  double m = 0.0;
  if (j < nj) {
    int64_t k = k0 + w;
    for (; k + 4 * 15 < ke; k += 4 * 16) {
      double v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = B[(k + 4 * u) * nj + j];
#pragma unroll
      for (int u = 0; u < 16; ++u) m = fmax(m, fabs(v[u]));
    }
    for (; k < ke; k += 4) m = fmax(m, fabs(B[k * nj + j]));
  }
  red[w * 64 + lane] = m;
  __syncthreads();
  if (w == 0 && j < nj) {
    m = fmax(fmax(red[lane], red[64 + lane]), fmax(red[128 + lane], red[192 + lane]));
    out[j] = m != 0.0 ? exponent_of(m) : INT32_MIN;
  }
}

constexpr int64_t kChunkRows = 512;

// Both in one launch: B's column exponents need none of A's work, and neither
// fills the memory by itself.  (On two streams, joined by events, they cost a
// call 10 us more at 1000 x 1000 x 1200 and no less at 4096^3.)  `chunks` parts
// of B's rows leave their exponents in part[chunk][njp] for split_cols_kernel.
__global__ __launch_bounds__(256) void prepare_kernel(const double* __restrict__ A, const double* __restrict__ B,
                                                      int64_t ni, int64_t nj, int64_t nk, int64_t nkp, int64_t nip,
                                                      int64_t njp, int64_t chunk_rows, int64_t column_blocks,
                                                      signed char* __restrict__ As, int* __restrict__ ea,
                                                      int* __restrict__ part, const CrtParams P) {
  __shared__ double red[256];
  const int64_t b = blockIdx.x;
  if (b < column_blocks) {
    const int64_t groups = njp / 64, chunk = b / groups, k0 = chunk * chunk_rows;
    const int64_t ke = k0 + chunk_rows < nk ? k0 + chunk_rows : nk;
    column_exponents(B, b % groups * 64, k0, ke, nj, part + chunk * njp, red);
  } else {
    split_row(A, b - column_blocks, ni, nk, nkp, nip, As, ea, P, red);
  }
}

// B -> Bs[t][j][k]: a workgroup owns 64 columns x 128 k; work-item (w, j)
// reads k0 + 16w .. k0 + 16w + 15 of column j (each load is 64 consecutive
// columns of one row) and, per modulus, packs those 16 residues into one
// 16-byte LDS write at row j, chunk w (rows padded to 144 bytes: the 16
// writes of a quarter-wavefront fall in distinct bank groups).  Eight
// work-items then read one 128-byte row back and store it as a whole line
// of Bs, so every store instruction writes eight whole lines.
constexpr int kColPitch = 144;  // bytes per LDS row of the B transpose
__global__ __launch_bounds__(512) void split_cols_kernel(const double* __restrict__ B, int64_t nk, int64_t nj,
                                                         int64_t nkp, int64_t njp, const int* __restrict__ part,
                                                         int chunks, int* __restrict__ fb,
                                                         signed char* __restrict__ Bs, const CrtParams P) {
  __shared__ __attribute__((aligned(16))) signed char lds[2][64 * kColPitch];
  const int tid = threadIdx.x;
  const int64_t j0 = int64_t(blockIdx.x) * 64;
  const int64_t j = j0 + (tid & 63);
  const int64_t kb = int64_t(blockIdx.y) * 128;
  const int64_t k0 = kb + 16 * (tid >> 6);
  int f = INT32_MIN;
  if (j < nj) {
    for (int c = 0; c < chunks; ++c) {
      const int e = part[c * njp + j];
      f = e > f ? e : f;
    }
    if (blockIdx.y == 0 && tid < 64) fb[j] = f;
  }
  const int sh = P.b - (f == INT32_MIN ? 0 : f);
  double x[16];
  if (j < nj && k0 + 16 <= nk) {
#pragma unroll
    for (int u = 0; u < 16; ++u) x[u] = B[(k0 + u) * nj + j];
  } else {
#pragma unroll
    for (int u = 0; u < 16; ++u) x[u] = (j < nj && k0 + u < nk) ? B[(k0 + u) * nj + j] : 0.0;
  }
  unsigned low[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    x[u] = rint(ldexp(x[u], sh));
    low[u] = low_word(x[u]);
  }
  const int jj = tid & 63, w16 = 16 * (tid >> 6);  // this work-item's LDS row and byte offset in it
  const int rrow = tid >> 3, rpart = 16 * (tid & 7);  // the row chunk it stores
  for (int t = 0; t < P.T; ++t) {
    v4i w;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      unsigned r[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q] = sym_mod(x[4 * c + q], low[4 * c + q], P.inv[t], P.minus_m[t]);
      w[c] = int(pack4(r[0], r[1], r[2], r[3]));
    }
    signed char* buf = lds[t & 1];
    *reinterpret_cast<v4i*>(buf + jj * kColPitch + w16) = w;
    __syncthreads();  // the row is complete; buffer t & 1 was last read two moduli ago, before the previous barrier
    const v4i row = *reinterpret_cast<const v4i*>(buf + rrow * kColPitch + rpart);
    *reinterpret_cast<v4i*>(Bs + (int64_t(t) * njp + j0 + rrow) * nkp + kb + rpart) = row;
  }
}

// LDS slot (in 16-byte chunks) of chunk c of tile row r; the XOR stays
// inside the row's kChunks slots.  It spreads the 16 rows an MFMA fragment
// reads at one chunk over all 16 bank groups (16-byte groups of a 256-byte
// bank cycle), and the chunks a loader wavefront writes likewise.
__device__ __forceinline__ int swz(int r, int c) {
  if constexpr (kChunks == 16) return r * kChunks + (c ^ (r & 15));
  else return r * kChunks + (c ^ ((r >> 1) & (kChunks - 1)));
}
static_assert(kChunks == 16 || kChunks == 8, "swizzle covers 8 or 16 chunks per row");

// 256x256 output tile per workgroup of eight wavefronts (64x128 each, a 4x8
// grid of 16x16 int32 accumulators).  For each modulus the K loop runs over
// that modulus's residues, and the epilogue reduces each exact int32 sum
// modulo m_t and stores the byte.  The tile size is set by L2 bandwidth: a
// stage brings 128 bytes of K for 256 rows of A and of B (64 KiB) for
// 8.4 M MACs, 128 MACs per byte, where a 128x128 tile's 64 left the MFMAs
// waiting on L2.  Two stages of LDS (128 KiB), one workgroup per CU.
constexpr int kThreads = 512;
constexpr int kWaveM = 64, kWaveN = 128;
constexpr int kFm = kWaveM / 16, kFn = kWaveN / 16;  // 16x16 tiles per wavefront
constexpr int kFrags = (kThreads / kWave) * kFm * kFn;  // accumulator fragments per workgroup tile
static_assert(kTM == kTN && kTM == 256 && kChunks == 8, "the stage loader covers 256 rows of 8 chunks");

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

// Stages go from global memory straight into LDS (global_load_lds, 16
// bytes per lane: each instruction fills 64 consecutive slots, i.e. 8
// swizzled rows, so lane l loads the logical chunk that swz() puts in slot
// l), one stage ahead of the one being computed.  All stages of all moduli
// form one sequence g = t * ksteps + st, so the next modulus's first stage
// is loaded during the current modulus's last.  The two stage buffers are
// separate arrays and the loop is unrolled by two, so every LDS access
// names its buffer: the compiler then sees that the loads in flight cannot
// write what the fragment reads read, and adds no wait for them; the wait
// for a stage is explicit (vmcnt(0), then the barrier that also frees the
// other buffer).  Against register-staged stages (loads into registers,
// then LDS stores a step later) this saves 32 VGPRs and the LDS store
// instructions: 1.05-1.06 against 1.08-1.10 ms per 4096^3 call.
__global__ __launch_bounds__(kThreads) void ozaki_gemm_kernel(unsigned* __restrict__ R,
                                                              const signed char* __restrict__ As,
                                                              const signed char* __restrict__ Bs, int64_t nip,
                                                              int64_t njp, int64_t nkp, int tiles_n, int per_group,
                                                              const CrtParams P) {
  __shared__ v4i A0[kTM * kChunks], A1[kTM * kChunks];
  __shared__ v4i B0[kTN * kChunks], B1[kTN * kChunks];
  int64_t tm, tn;
  tile_of(blockIdx.x, gridDim.x, int(nip / kTM), tiles_n, tm, tn);
  const int64_t m0 = tm * kTM, n0 = tn * kTN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * kWaveM, wn = (wave & 1) * kWaveN;
  const int ksteps = int(nkp / kTK);  // even: nkp is a multiple of 2 kTK
  const int t_begin = int(blockIdx.y) * per_group;  // this workgroup's moduli
  const int t_end = t_begin + per_group < P.T ? t_begin + per_group : P.T;
  const int total = t_end * ksteps;  // the stage after its last
  const int fr = lane & 15, fk = lane >> 4;  // MFMA operand row and k quarter
  // This wavefront's fragments in the residue array: [tile][wave][i][j][lane].
  const int64_t frag0 = ((tm * tiles_n + tn) * (kThreads / kWave) + wave) * (kFm * kFn);
  const int64_t per_mod = nip * njp / 4;  // 32-bit words per modulus
  // Loader: instruction u (0..3) of wavefront w fills slots 64 (4w + u) ..
  // + 63: row drow0 + 8u (drow0 = 32w + lane/8), physical chunk lane%8,
  // which holds logical chunk (lane%8) ^ ((row >> 1) & 7).
  const int drow0 = 32 * wave + (lane >> 3);
  int dchunk[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) dchunk[u] = (lane & 7) ^ (((drow0 + 8 * u) >> 1) & 7);
  const signed char* a0 = As + (m0 + drow0) * nkp;
  const signed char* b0 = Bs + (n0 + drow0) * nkp;
  const int64_t a_mod = nip * nkp, b_mod = njp * nkp;
  auto load_stage = [&](int g, v4i* Ad, v4i* Bd) {  // stage g: modulus g / ksteps, K step g % ksteps
    const int tt = g / ksteps, st = g - tt * ksteps;
    const signed char* at = a0 + tt * a_mod + st * kTK;
    const signed char* bt = b0 + tt * b_mod + st * kTK;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      __builtin_amdgcn_global_load_lds((global_void*)(at + int64_t(8 * u) * nkp + 16 * dchunk[u]),
                                       (lds_void*)(Ad + 64 * (4 * wave + u)), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((global_void*)(bt + int64_t(8 * u) * nkp + 16 * dchunk[u]),
                                       (lds_void*)(Bd + 64 * (4 * wave + u)), 16, 0, 0);
    }
  };
  v4i acc[kFm][kFn];
  auto compute = [&](const v4i* Ar, const v4i* Br) {
    // Raised wave priority over the MFMA block: with two wavefronts per
    // SIMD the arbiter then keeps feeding the matrix pipe from one while
    // the other issues its loads.
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kk = 0; kk < kChunks / 4; ++kk) {
      const int c = kk * 4 + fk;
      v4i af[kFm], bf[kFn];
#pragma unroll
      for (int i = 0; i < kFm; ++i) af[i] = Ar[swz(wm + i * 16 + fr, c)];
#pragma unroll
      for (int j = 0; j < kFn; ++j) bf[j] = Br[swz(wn + j * 16 + fr, c)];
#pragma unroll
      for (int i = 0; i < kFm; ++i)
#pragma unroll
        for (int j = 0; j < kFn; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[i], bf[j], acc[i][j], 0, 0, 0);
      // The backend's LDS-read/MFMA interleave for small GEMM loops: 1.056-1.063
      // against 1.085-1.093 ms per 4096^3 call, alternating runs (an explicit
      // one LDS read per two MFMAs was slower, 1.10 ms).
      __builtin_amdgcn_iglp_opt(0);
    }
    __builtin_amdgcn_s_setprio(0);
  };
  // This wavefront's stage loads have landed (vmcnt(0)); after the barrier
  // every wavefront's have, and every wavefront has finished reading the
  // other buffer (its reads fed the MFMAs issued before the barrier).
  auto stage_ready = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  int g = t_begin * ksteps;
  load_stage(g, A0, B0);
  for (int t = t_begin; t < t_end; ++t) {
#pragma unroll
    for (int i = 0; i < kFm; ++i)
#pragma unroll
      for (int j = 0; j < kFn; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    for (int st = 0; st < ksteps; st += 2, g += 2) {
      stage_ready();  // stage g in buffer 0
      if (g + 1 < total) load_stage(g + 1, A1, B1);
      compute(A0, B0);
      stage_ready();  // stage g + 1 in buffer 1
      if (g + 2 < total) load_stage(g + 2, A0, B0);
      compute(A1, B1);
    }
    // d_t = the sum's symmetric residue modulo m_t (|sum| < 2^31, see
    // sym_mod); the four rows of a lane's accumulator go to one 32-bit word.
    const double inv = P.inv[t];
    const unsigned minus_m = P.minus_m[t];
    unsigned* rt = R + int64_t(t) * per_mod + frag0 * kWave + lane;
#pragma unroll
    for (int i = 0; i < kFm; ++i)
#pragma unroll
      for (int j = 0; j < kFn; ++j) {
        unsigned d[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) d[r] = sym_mod(double(acc[i][j][r]), unsigned(acc[i][j][r]), inv, minus_m);
        rt[(i * kFn + j) * kWave] = pack4(d[0], d[1], d[2], d[3]);
      }
  }
}

// One work-item per (fragment, lane): the four outputs of that accumulator
// slot.  X/M = sum_t d_t (h_t + l_t) mod 1; the h_t part is exact (every
// term is a multiple of 2^-44 below 128 in magnitude, and the sum is reduced
// modulo 1 after every three: below 385, it is a 53-bit multiple of 2^-44).
// T is a template parameter: with it as a variable the loop over the moduli
// was not unrolled and indexed the words through the index register (13 moduli,
// 1000 x 1000: 8.0 us, 6.0 here; 4096 x 4096: 76 us both, 54 for the 13 bytes
// in and 8 out of an element).
template <int T>
__global__ __launch_bounds__(256) void crt_combine_kernel(double* __restrict__ C, const unsigned* __restrict__ R,
                                                          const int* __restrict__ ea, const int* __restrict__ fb,
                                                          double alpha, double beta, int use_beta, int64_t ni,
                                                          int64_t nj, int64_t nip, int64_t njp, int tiles_n,
                                                          const CrtParams P) {
  const int64_t g = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int64_t per_mod = nip * njp / 4;
  if (g >= per_mod) return;
  const int lane = int(g % kWave);
  const int64_t frag = g / kWave;
  const int64_t tile = frag / kFrags;
  const int f = int(frag % kFrags);
  const int wave = f / (kFm * kFn), i = (f / kFn) % kFm, j = f % kFn;
  const int64_t row0 = (tile / tiles_n) * kTM + (wave >> 1) * kWaveM + i * 16 + 4 * (lane >> 4);
  const int64_t col = (tile % tiles_n) * kTN + (wave & 1) * kWaveN + j * 16 + (lane & 15);
  // All residue words first, so their loads are in flight together.
  unsigned wv[T];
#pragma unroll
  for (int t = 0; t < T; ++t) wv[t] = R[int64_t(t) * per_mod + g];
  double fh[4] = {0.0, 0.0, 0.0, 0.0}, fl[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const double h = P.h[t], l = P.l[t];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double d = double(int(wv[t] << (24 - 8 * r)) >> 24);  // the signed byte r
      fh[r] = fma(d, h, fh[r]);
      if (t % 3 == 2) fh[r] = __builtin_amdgcn_fract(fh[r]);
      fl[r] = fma(d, l, fl[r]);
    }
  }
  if (col >= nj) return;
  const int fj = fb[col];
  const int sc = (fj == INT32_MIN ? 0 : fj) - 2 * P.b;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t row = row0 + r;
    if (row >= ni) break;
    // X = (fx + fl) M with fx = fh - nearest integer (exact, a multiple of
    // 2^-52 in [-1/2, 1/2]) and M = M_hi + M_lo: the product fx M_hi is
    // split exactly by an fma, the small terms are added to its error.
    const double f1 = __builtin_amdgcn_fract(fh[r]);
    double fx = f1 - rint(f1);
    if (fx + fl[r] > 0.5) fx -= 1.0;
    if (fx + fl[r] < -0.5) fx += 1.0;
    const double p = fx * P.M_hi;
    const double e = fma(fx, P.M_hi, -p);
    const double x = p + (e + fma(fx, P.M_lo, fl[r] * P.M_hi));
    const double v = alpha * ldexp(x, ea[row] + sc);
    double* c = C + row * nj + col;
    *c = use_beta ? v + beta * *c : v;
  }
}

template <int T = 1, class... Args>
void launch_combine(int moduli, dim3 grid, hipStream_t s, const Args&... args) {
  if (moduli == T) crt_combine_kernel<T><<<grid, dim3(256), 0, s>>>(args...);
  else if constexpr (T < kMaxMods) launch_combine<T + 1>(moduli, grid, s, args...);
}

// Moduli per workgroup.  With all T in one, the tiles of a small C leave most
// CUs idle (512^3 on four workgroups: 135 us a call, 28 on 52; 2048^3 on 64:
// 400 us, 178 on 256); each modulus is a GEMM of its own,
// so they go to as many workgroups as make the fewest stages in a row.  A
// workgroup costs about two stages besides (its first loads, its launch), and
// more rounds of 256 workgroups are taken only for fewer stages.
int moduli_per_group(int64_t tiles, int T, int64_t ksteps) {
  int best = T;
  int64_t least = INT64_MAX;
  for (int per = T; per >= 1; --per) {
    const int64_t stages = ceil_div(tiles * ceil_div(T, per), int64_t(256)) * (per * ksteps + 2);
    if (stages < least) least = stages, best = per;
  }
  return best;
}

}  // namespace

extern "C" {

size_t rpx_gemm_mixed_scratch_bytes(int64_t ni, int64_t nj, int64_t nk, int nmoduli) {
  if (ni < 0 || nj < 0 || nk < 0 || nmoduli < 0 || nmoduli > kMaxMods || nk > kMaxK) return 0;
  CrtParams P;
  if (!crt_setup(nk, nmoduli, &P)) return 0;
  return mixed_layout(ni, nj, nk, P.T).total;
}

int rpx_gemm_mixed_bits(int64_t nk, int nmoduli) {
  if (nk < 0 || nk > kMaxK || nmoduli < 0 || nmoduli > kMaxMods) return RPX_ERR_INVALID_ARGUMENT;
  CrtParams P;
  if (!crt_setup(nk, nmoduli, &P)) return RPX_ERR_UNSUPPORTED;
  return P.b;
}

int rpx_gemm_mixed_f64(double* C, const double* A, const double* B, double alpha, double beta, int64_t ni,
                       int64_t nj, int64_t nk, int nmoduli, void* scratch, size_t scratch_bytes, void* stream) {
  return rpx_gemm_mixed_tuned_f64(C, A, B, alpha, beta, ni, nj, nk, nmoduli, nullptr, scratch, scratch_bytes,
                                  stream);
}

int rpx_gemm_mixed_tuned_f64(double* C, const double* A, const double* B, double alpha, double beta, int64_t ni,
                             int64_t nj, int64_t nk, int nmoduli, const rpx_tuning* tune, void* scratch,
                             size_t scratch_bytes, void* stream) {
  if (ni < 0 || nj < 0 || nk < 0 || nmoduli < 0 || nmoduli > kMaxMods) return RPX_ERR_INVALID_ARGUMENT;
  if (ni == 0 || nj == 0) return RPX_SUCCESS;
  if (!C || !scratch || (nk > 0 && (!A || !B))) return RPX_ERR_INVALID_ARGUMENT;
  if (nk > kMaxK) return RPX_ERR_UNSUPPORTED;
  CrtParams P;
  if (!crt_setup(nk, nmoduli, &P)) return RPX_ERR_UNSUPPORTED;
  const MixedLayout l = mixed_layout(ni, nj, nk, P.T);
  if (scratch_bytes < l.total) return RPX_ERR_SCRATCH_TOO_SMALL;
  const int64_t tm = l.nip / kTM, tn = l.njp / kTN;
  if (l.nip + l.njp > INT32_MAX || tm * tn > INT32_MAX || ceil_div(l.nip * l.njp / 4, 256) > INT32_MAX)
    return RPX_ERR_UNSUPPORTED;
  char* base = reinterpret_cast<char*>(scratch);
  signed char* As = reinterpret_cast<signed char*>(base + l.a_off);
  signed char* Bs = reinterpret_cast<signed char*>(base + l.b_off);
  int* ea = reinterpret_cast<int*>(base + l.ea_off);
  int* fb = reinterpret_cast<int*>(base + l.fb_off);
  unsigned* R = reinterpret_cast<unsigned*>(base + l.r_off);
  hipStream_t s = as_stream(stream);
  // The column exponents' parts lie where the residue bytes d_t go later.
  int* part = reinterpret_cast<int*>(base + l.r_off);
  const int64_t chunks = nk > 0 ? std::min(ceil_div(nk, kChunkRows), int64_t(kTM / 4)) : 0;
  const int64_t chunk_rows = chunks > 0 ? ceil_div(nk, chunks) : 0, column_blocks = chunks * (l.njp / 64);
  prepare_kernel<<<dim3(unsigned(column_blocks + l.nip)), dim3(256), 0, s>>>(
      A, B, ni, nj, nk, l.nkp, l.nip, l.njp, chunk_rows, column_blocks, As, ea, part, P);
  split_cols_kernel<<<dim3(unsigned(l.njp / 64), unsigned(l.nkp / 128)), dim3(512), 0, s>>>(
      B, nk, nj, l.nkp, l.njp, part, int(chunks), fb, Bs, P);
  const int per_group = moduli_per_group(tm * tn, P.T, l.nkp / kTK);
  ozaki_gemm_kernel<<<dim3(unsigned(tm * tn), unsigned(ceil_div(P.T, per_group))), dim3(kThreads), 0, s>>>(
      R, As, Bs, l.nip, l.njp, l.nkp, int(tn), per_group, P);
  const int use_beta = (tune_flags(tune) & RPX_TUNE_GEMM_BETA) != 0;
  const dim3 combine(unsigned(ceil_div(l.nip * l.njp / 4, 256)));
  launch_combine(P.T, combine, s, C, R, ea, fb, alpha, beta, use_beta, ni, nj, l.nip, l.njp, int(tn), P);
  return launch_status();
}

}  // extern "C"
