// GEMM (polybench): C[i][j] = sum_k (alpha*A[i][k]) * B[k][j].  With
// RPX_TUNE_GEMM_BETA the textbook form C = alpha*A*B + beta*C instead (the
// old C read once and beta*C added to the finished sum).
//
// Reference: src/polybench/POLYBENCH_GEMM.hpp:12-50 (C *= beta, then C is
// overwritten by the dot, so beta never reaches the result),
// POLYBENCH_GEMM-Seq.cpp:30-50, POLYBENCH_GEMM-Hip.cpp:27-102 (one thread
// per C element, no LDS, no matrix cores).
//
// Two FP64 paths:
//  * gemm_naive_kernel: the one-thread-per-element shape of the suite's
//    Base_HIP variant, kept as the "plain FP64 GPU" comparator;
//  * gemm_mfma_f64_kernel: v_mfma_f64_16x16x4f64 on workgroup tiles from
//    128 x 128 to 16 x 16, by size; tiles are mapped XCD-major so neighbouring
//    tiles that share A rows / B columns run on the same XCD's L2.
#include <cmath>
#include <type_traits>

#include "rpx_common.hpp"

using namespace rpx;

namespace {

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));

// ---- plain FP64 comparator ---------------------------------------------------
__global__ __launch_bounds__(256) void gemm_naive_kernel(double* __restrict__ C, const double* __restrict__ A,
                                                         const double* __restrict__ B, double alpha, double beta,
                                                         int use_beta, int64_t ni, int64_t nj, int64_t nk) {
  const int64_t j = int64_t(blockIdx.x) * 32 + (threadIdx.x & 31);
  const int64_t i = int64_t(blockIdx.y) * 8 + (threadIdx.x >> 5);
  if (i >= ni || j >= nj) return;
  double dot = 0.0;
  for (int64_t k = 0; k < nk; ++k) dot = fma(alpha * A[k + i * nk], B[j + k * nj], dot);
  C[j + i * nj] = use_beta ? dot + beta * C[j + i * nj] : dot;
}

// ---- FP64 MFMA ---------------------------------------------------------------
//
// A workgroup computes a tile of C with WM x WN x WK wavefronts: each owns
// MF x NF tiles of v_mfma_f64_16x16x4f64 and, of every K slab, the WK-th part
// of TK deep (partial sums of the WK groups meet in LDS at the end, added in
// a fixed order).  Slabs are double-buffered in LDS, both operands
// k-contiguous ([m][k] for A, [n][k] for B, rows padded by two doubles); in
// each pair of MFMA steps lane (r, q) of a fragment takes the adjacent
// k = 8h + 2q and 8h + 2q + 1, so one 16-byte LDS read feeds two MFMAs.  The
// k order inside a slab is thereby permuted; the result is the same sum in
// another association.  The next slab's global loads are in flight during the
// current slab's MFMAs and nothing reads them before those are issued: A is
// scaled by alpha, as the suite rounds alpha*A[i][k], on its way to LDS.
// Rows and columns outside C are loaded from its last ones (their products are
// never stored); only the K remainder is zeroed.
typedef v2d v2d_u __attribute__((aligned(8)));

template <int MF_, int NF_, int WM_, int WN_, int WK_, int TK_, int FB_>
struct Shape {
  static constexpr int FB = FB_;  // fragment sets: 2 where the registers allow reading a step ahead
  static constexpr int MF = MF_, NF = NF_, WM = WM_, WN = WN_, WK = WK_, TK = TK_;
  static constexpr int TM = 16 * MF * WM, TN = 16 * NF * WN, KS = TK * WK, T = kWave * WM * WN * WK;
  static constexpr int LR = KS + 2;              // doubles per LDS row of either operand
  static constexpr int PA = TM * KS / 2 / T;     // 16-byte pairs of A per work-item and slab
  static constexpr int PB = TN * KS / 4 / T;     // 2x2 blocks of B
  static constexpr int kSlabs = 2 * (TM + TN) * LR, kSums = WK > 1 ? WK * TM * TN : 0;
  static constexpr int kLds = kSlabs > kSums ? kSlabs : kSums;
  static_assert(PA * T * 2 == TM * KS && PB * T * 4 == TN * KS, "whole pairs and blocks");
  static_assert(TK % 8 == 0, "whole steps");
};

// INF: alpha is infinite, and the zeros beyond K are put in after the scaling,
// which makes NaNs of them.  A kernel of its own because the test in the loop
// costs the others 1.5 to 4% (1000 x 1000 x 1200: 51.9 -> 52.7 us at best).
template <typename S, bool INF>
__global__ __launch_bounds__(S::T, 2) void gemm_mfma_f64_kernel(double* __restrict__ C, const double* __restrict__ A,
                                                             const double* __restrict__ B, double alpha, double beta,
                                                             int use_beta, int64_t ni, int64_t nj, int64_t nk,
                                                             int tiles_n) {
  __shared__ __attribute__((aligned(16))) double lds[S::kLds];
  auto As = [&](int buf) { return lds + buf * S::TM * S::LR; };
  auto Bs = [&](int buf) { return lds + 2 * S::TM * S::LR + buf * S::TN * S::LR; };

  const unsigned tile = xcd_major(blockIdx.x, gridDim.x);
  const int64_t m0 = int64_t(tile / unsigned(tiles_n)) * S::TM;
  const int64_t n0 = int64_t(tile % unsigned(tiles_n)) * S::TN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % S::WN * 16 * S::NF, wm = wave / S::WN % S::WM * 16 * S::MF, wk = wave / (S::WN * S::WM);
  const bool n_inside = n0 + S::TN <= nj;

  const double* pa[S::PA];  // this work-item's row of A, at its k
  int ka[S::PA];
  const double* pb[S::PB];  // its first row of B, first column
  int kb[S::PB], nb[S::PB], odd[S::PB];
#pragma unroll
  for (int u = 0; u < S::PA; ++u) {
    const int at = tid + u * S::T;
    const int64_t row = m0 + at / (S::KS / 2);
    ka[u] = 2 * (at % (S::KS / 2));
    pa[u] = A + (row < ni ? row : ni - 1) * nk + ka[u];
  }
#pragma unroll
  for (int u = 0; u < S::PB; ++u) {
    const int at = tid + u * S::T;
    nb[u] = 2 * (at % (S::TN / 2));
    kb[u] = 2 * (at / (S::TN / 2));
    const int64_t c = n0 + nb[u];
    odd[u] = c + 1 < nj;  // the second column exists
    pb[u] = B + kb[u] * nj + (c < nj ? c : nj - 1);
  }
  v2d ra[S::PA], rb[S::PB][2];
  auto load_slab = [&](int64_t k0) {
    if (k0 + S::KS <= nk) {
#pragma unroll
      for (int u = 0; u < S::PA; ++u) ra[u] = *reinterpret_cast<const v2d_u*>(pa[u] + k0);
      if (n_inside) {
#pragma unroll
        for (int u = 0; u < S::PB; ++u)
#pragma unroll
          for (int t = 0; t < 2; ++t) rb[u][t] = *reinterpret_cast<const v2d_u*>(pb[u] + (k0 + t) * nj);
      } else {
#pragma unroll
        for (int u = 0; u < S::PB; ++u)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            rb[u][t].x = pb[u][(k0 + t) * nj];
            rb[u][t].y = pb[u][(k0 + t) * nj + odd[u]];
          }
      }
    } else {  // the K remainder
      const int left = int(nk - k0);
#pragma unroll
      for (int u = 0; u < S::PA; ++u) {
        ra[u].x = ka[u] < left ? pa[u][k0] : 0.0;
        ra[u].y = ka[u] + 1 < left ? pa[u][k0 + 1] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < S::PB; ++u)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          rb[u][t].x = kb[u] + t < left ? pb[u][(k0 + t) * nj] : 0.0;
          rb[u][t].y = kb[u] + t < left ? pb[u][(k0 + t) * nj + odd[u]] : 0.0;
        }
    }
  };
  auto store_slab = [&](int buf, int64_t k0) {
#pragma unroll
    for (int u = 0; u < S::PA; ++u) {
      v2d a = alpha * ra[u];
      if constexpr (INF) {
        a.x = k0 + ka[u] < nk ? a.x : 0.0;
        a.y = k0 + ka[u] + 1 < nk ? a.y : 0.0;
      }
      *reinterpret_cast<v2d*>(As(buf) + (tid + u * S::T) / (S::KS / 2) * S::LR + ka[u]) = a;
    }
#pragma unroll
    for (int u = 0; u < S::PB; ++u) {
      *reinterpret_cast<v2d*>(Bs(buf) + nb[u] * S::LR + kb[u]) = v2d{rb[u][0].x, rb[u][1].x};
      *reinterpret_cast<v2d*>(Bs(buf) + (nb[u] + 1) * S::LR + kb[u]) = v2d{rb[u][0].y, rb[u][1].y};
    }
  };

  v4d acc[S::MF][S::NF];
#pragma unroll
  for (int i = 0; i < S::MF; ++i)
#pragma unroll
    for (int j = 0; j < S::NF; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

  const int fr = lane & 15;  // fragment row (A) / column (B)
  const int fk = wk * S::TK + 2 * (lane >> 4);
  v2d af[S::FB][S::MF], bf[S::FB][S::NF];
  auto read_frags = [&](int buf, int h, int to) {
#pragma unroll
    for (int i = 0; i < S::MF; ++i)
      af[to][i] = *reinterpret_cast<const v2d*>(As(buf) + (wm + i * 16 + fr) * S::LR + 8 * h + fk);
#pragma unroll
    for (int j = 0; j < S::NF; ++j)
      bf[to][j] = *reinterpret_cast<const v2d*>(Bs(buf) + (wn + j * 16 + fr) * S::LR + 8 * h + fk);
  };
  // A step is two halves, the first k of every lane and the second, so each
  // accumulator's two MFMAs are apart.  With two fragment sets the next step's
  // are read between the halves; the slab's last step then runs behind the
  // barrier, over the first reads of the next slab.
  constexpr int kSteps = S::TK / 8;
  static_assert(S::FB == 1 || kSteps % 2 == 0, "a slab begins with set 0");
  if (nk > 0) {
    load_slab(0);
    store_slab(0, 0);
    __syncthreads();
    if (S::FB == 2) read_frags(0, 0, 0);
  }
  int buf = 0;
  for (int64_t k0 = 0; k0 < nk; k0 += S::KS) {
    const bool more = k0 + S::KS < nk;
    if (more) load_slab(k0 + S::KS);
#pragma unroll
    for (int h = 0; h < kSteps; ++h) {
      const int cur = S::FB == 2 ? h % 2 : 0, nxt = S::FB == 2 ? cur ^ 1 : 0;
      if (S::FB == 1) read_frags(buf, h, 0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < S::MF; ++i)
#pragma unroll
        for (int j = 0; j < S::NF; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[cur][i].x, bf[cur][j].x, acc[i][j], 0, 0, 0);
      if (S::FB == 2 && h + 1 < kSteps) read_frags(buf, h + 1, nxt);
      if (S::FB == 2 && h + 1 == kSteps && more) {
        store_slab(buf ^ 1, k0 + S::KS);
        __syncthreads();
        read_frags(buf ^ 1, 0, nxt);
      }
#pragma unroll
      for (int i = 0; i < S::MF; ++i)
#pragma unroll
        for (int j = 0; j < S::NF; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[cur][i].y, bf[cur][j].y, acc[i][j], 0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
    if (S::FB == 1 && more) {
      store_slab(buf ^ 1, k0 + S::KS);
      __syncthreads();
    }
    buf ^= 1;
  }

  // With beta the old values of a batch of elements are loaded before the first
  // of them is stored: each load would otherwise wait for the store before it
  // (500^3 with beta and the copy of C: 14.9 us, 13.9 here).
  auto old = [&](int64_t gi, int64_t gj) { return use_beta && gi < ni && gj < nj ? C[gi * nj + gj] : 0.0; };
  auto put = [&](int64_t gi, int64_t gj, double v, double c) {
    if (gi < ni && gj < nj) C[gi * nj + gj] = use_beta ? fma(beta, c, v) : v;
  };
  // v_mfma_f64_16x16x4f64 accumulator layout (measured on gfx950): element r
  // of lane l is row 4*r + l/16, column l%16.
  if constexpr (S::WK == 1) {
    const int64_t row0 = m0 + wm + (lane >> 4), col0 = n0 + wn + fr;
    // A tile inside C of a shape for short K, which the stores bound: without
    // a test for each element.  (Big has no registers left for it: 4096^2 x
    // 1024 539 -> 566 us.)
    if (S::FB == 1 && m0 + S::TM <= ni && n_inside) {
      double* to = C + row0 * nj + col0;
#pragma unroll
      for (int i = 0; i < S::MF; ++i) {
        double c[S::NF][4];
        if (use_beta) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < S::NF; ++j) c[j][r] = to[(i * 16 + 4 * r) * nj + j * 16];
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < S::NF; ++j) to[(i * 16 + 4 * r) * nj + j * 16] = fma(beta, c[j][r], acc[i][j][r]);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < S::NF; ++j) to[(i * 16 + 4 * r) * nj + j * 16] = acc[i][j][r];
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < S::MF; ++i) {
      double c[S::NF][4];
#pragma unroll
      for (int j = 0; j < S::NF; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) c[j][r] = old(row0 + i * 16 + 4 * r, col0 + j * 16);
#pragma unroll
      for (int j = 0; j < S::NF; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) put(row0 + i * 16 + 4 * r, col0 + j * 16, acc[i][j][r], c[j][r]);
    }
  } else {
    constexpr int kPer = (S::TM * S::TN + S::T - 1) / S::T;  // elements per work-item
    double c[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int e = tid + u * S::T;
      c[u] = e < S::TM * S::TN ? old(m0 + e / S::TN, n0 + e % S::TN) : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < S::MF; ++i)
#pragma unroll
      for (int j = 0; j < S::NF; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          lds[(wk * S::TM + wm + i * 16 + 4 * r + (lane >> 4)) * S::TN + wn + j * 16 + fr] = acc[i][j][r];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int e = tid + u * S::T;
      if (e >= S::TM * S::TN) continue;
      double v = lds[e];
#pragma unroll
      for (int k = 1; k < S::WK; ++k) v += lds[k * S::TM * S::TN + e];
      put(m0 + e / S::TN, n0 + e % S::TN, v, c[u]);
    }
  }
}

template <typename S, bool INF = false>
int launch_mfma(double* C, const double* A, const double* B, double alpha, double beta, int use_beta, int64_t ni,
                int64_t nj, int64_t nk, hipStream_t s) {
  const int64_t tm = ceil_div(ni, S::TM), tn = ceil_div(nj, S::TN);
  if (tm * tn > INT32_MAX || tn > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  gemm_mfma_f64_kernel<S, INF><<<dim3(unsigned(tm * tn)), dim3(S::T), 0, s>>>(C, A, B, alpha, beta, use_beta, ni, nj, nk,
                                                                       int(tn));
  return launch_status();
}

// The shapes, largest tile first.  A large tile moves the least data per
// product, but C has to hold 256 tiles before every CU has one; small tiles
// split K over their wavefronts instead, so that few of them still fill the
// matrix cores.
//
// What bounds them: FP64 MFMA issue, 64 clocks each (77 TF/s, measured), and
// how evenly the tiles go over 256 CUs.  4096^3 runs at 66.7 TF/s (2.06 ms) on
// sixteen wavefronts of 32 x 32 with slabs 32 deep; four wavefronts of 64 x 64,
// slabs of 16 and two workgroups per CU took 2.14 ms, and as a lone tile kept
// half of a SIMD's time: 2048^2 x 4096 612 -> 517 us, 4000 x 3000 x 2000
// 1054 -> 785.  1000 x 1000 x 1200 took 261 us as 64 tiles of 128 x 128 on 256
// CUs and takes 54 us as 256 tiles of 64 x 64 (31 us of MFMAs, 10 us of launch,
// first loads and epilogue, the rest LDS writes and loads).  Tiles of 96 x 96
// and 96 x 64 are for the sizes between: 1500^3 178 -> 129 us, 1100 x 1100 x
// 4000 268 -> 244.
using Big = Shape<2, 2, 4, 4, 1, 32, 2>;     // 128 x 128, sixteen wavefronts
using Short = Shape<1, 4, 4, 2, 1, 16, 1>;   // 64 x 128, eight wavefronts, two workgroups per CU, for short K
using Square = Shape<3, 2, 2, 3, 2, 16, 2>;  // 96 x 96, K in two, twelve wavefronts
using Tall = Shape<3, 2, 2, 2, 2, 16, 2>;    // 96 x 64, K in two, eight wavefronts
using Mid = Shape<2, 2, 2, 2, 2, 16, 2>;     // 64 x 64, K in two, two workgroups per CU
using MidDeep = Shape<2, 2, 2, 2, 4, 16, 2>; // 64 x 64, K in four, one workgroup per CU
using Small = Shape<2, 2, 1, 1, 4, 8, 1>;    // 32 x 32, K in four
using SmallDeep = Shape<2, 2, 1, 1, 8, 8, 1>;// 32 x 32, K in eight
using Tiny = Shape<1, 1, 1, 1, 8, 16, 1>;    // 16 x 16, K in eight

// Time of a product without the launch, in microseconds: a tile alone on a CU
// takes `alone` per unit of K, a CU's n-th tile `shared` (both fitted to 24
// sizes from 64^3 to 4096^3, within about 15%).
template <typename S>
double mfma_us(int64_t ni, int64_t nj, int64_t nk, double alone, double shared) {
  const double n = double(ceil_div(ni, S::TM)) * double(ceil_div(nj, S::TN)) / 256.0;
  const double per_k = shared * (n < 8 ? double(ceil_div(int64_t(n * 256.0), 256)) : n + 0.5);
  return double(ceil_div(nk, S::KS) * S::KS) * (per_k > alone ? per_k : alone);
}

// The same with what a tile costs besides: its first loads, its stores.
template <typename S>
double tiles_us(int64_t ni, int64_t nj, double tile) {
  return tile * double(ceil_div(ni, S::TM)) * double(ceil_div(nj, S::TN)) / 256.0;
}

int gemm_mfma(double* C, const double* A, const double* B, double alpha, double beta, int use_beta, int64_t ni,
              int64_t nj, int64_t nk, hipStream_t s) {
  if (__builtin_isinf(alpha)) return launch_mfma<Mid, true>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
  const double us[] = {mfma_us<Big>(ni, nj, nk, 0.126, 0.1255),        mfma_us<Square>(ni, nj, nk, 0.0845, 0.0835),
                       mfma_us<Tall>(ni, nj, nk, 0.0605, 0.0595),      mfma_us<Mid>(ni, nj, nk, 0.0435, 0.0365),
                       mfma_us<MidDeep>(ni, nj, nk, 0.0405, 0.039),    mfma_us<Small>(ni, nj, nk, 0.0163, 0.0122),
                       mfma_us<SmallDeep>(ni, nj, nk, 0.0138, 0.0122), mfma_us<Tiny>(ni, nj, nk, 0.0049, 0.0047)};
  int best = 0;
  for (int i = 1; i < 8; ++i)
    if (us[i] < us[best]) best = i;
  // Short tiles for a C of at least one per CU and K up to 300 or so, where a
  // tile costs 1.8 us besides its products and one of 128 x 128, alone on its
  // CU, 7 us: 4096^2 x 64 60.1 -> 51.7 us, x 128 91.5 -> 85.7, 8192^2 x 16
  // 166 -> 97, 1024 x 2048 x 16 9.5 -> 6.7.
  const double besides[] = {tiles_us<Big>(ni, nj, 7.0),     tiles_us<Square>(ni, nj, 5.0),
                            tiles_us<Tall>(ni, nj, 4.1),    tiles_us<Mid>(ni, nj, 2.1),
                            tiles_us<MidDeep>(ni, nj, 3.7), tiles_us<Small>(ni, nj, 0.54),
                            tiles_us<SmallDeep>(ni, nj, 0.9), tiles_us<Tiny>(ni, nj, 1.1)};
  const double n = tiles_us<Short>(ni, nj, 1.0);  // per CU
  const double rounds = n < 4 ? std::ceil(n) : n < 8 ? n + 0.25 : n;
  const double short_us = rounds * (double(ceil_div(nk, Short::KS) * Short::KS) * 0.0695 + 1.8);
  if (ni >= Short::TM && n >= 1 && short_us < 0.98 * (us[best] + besides[best]))
    return launch_mfma<Short>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
  switch (best) {
    case 0: return launch_mfma<Big>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
    case 1: return launch_mfma<Square>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
    case 2: return launch_mfma<Tall>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
    case 3: return launch_mfma<Mid>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
    case 4: return launch_mfma<MidDeep>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
    case 5: return launch_mfma<Small>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
    case 6: return launch_mfma<SmallDeep>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
    default: return launch_mfma<Tiny>(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
  }
}

}  // namespace

extern "C" {

int rpx_gemm_f64(double* C, const double* A, const double* B, double alpha, double beta, int64_t ni,
                 int64_t nj, int64_t nk, const rpx_tuning* tune, void* stream) {
  if (ni < 0 || nj < 0 || nk < 0) return RPX_ERR_INVALID_ARGUMENT;
  if (ni == 0 || nj == 0) return RPX_SUCCESS;
  if (!C || (nk > 0 && (!A || !B))) return RPX_ERR_INVALID_ARGUMENT;
  hipStream_t s = as_stream(stream);
  const int use_beta = (tune_flags(tune) & RPX_TUNE_GEMM_BETA) != 0;
  if (tune_flags(tune) & RPX_TUNE_NAIVE) {
    const int64_t gx = ceil_div(nj, 32), gy = ceil_div(ni, 8);
    if (gx > INT32_MAX || gy > 65535) return RPX_ERR_UNSUPPORTED;
    gemm_naive_kernel<<<dim3(unsigned(gx), unsigned(gy)), dim3(256), 0, s>>>(C, A, B, alpha, beta, use_beta, ni,
                                                                              nj, nk);
    return launch_status();
  }
  return gemm_mfma(C, A, B, alpha, beta, use_beta, ni, nj, nk, s);
}

}  // extern "C"
