// JACOBI_2D, several time steps per launch on one register-resident tile per
// workgroup.
//
// Reference: src/polybench/POLYBENCH_JACOBI_2D-Seq.cpp:30-54 (tsteps x two
// sweeps over the interior).
//
// A workgroup of W wavefronts holds W*RW rows of 128 columns: a lane holds
// the column pair 2*lane of RW consecutive rows, twice (the A and the B of the
// time step).  A sweep computes one array from the other; west and east
// neighbours come from the adjacent lanes (DPP moves), the rows above and
// below a wavefront's RW rows from LDS, with one barrier per sweep.  With
// `steps` time steps per launch the outer 2*steps rows and columns go stale and
// only the inside is stored; tiles at the grid's edge start on it and keep its
// boundary cells, so they have no halo on that side.  Boundary cells are
// always read from A and B themselves, so the grid the launches ping-pong
// through needs no boundary.  Rows of odd N start on 8 bytes only; the
// 16-byte loads and stores here do not need more.
//
// What bounds it: FP64 issue.  A row and sweep of a wavefront is 10 FP64
// instructions and 4 DPP moves, measured 4.5-4.7 and 4.3 clocks each, so 64
// clocks; a sweep of a 64-row tile alone on a CU takes 0.53 us (0.43 us at
// that rate, the rest barrier and LDS), a launch about 4 us besides.
// N = 1002, 40 time steps: 374 us with the 16-row wavefront tiles of
// jacobi_fused_kernel (13 launches of 27 us, each one wavefront's serial
// chain of 28 rows x 6 levels), 82 us here (7 launches).  N = 8192, 50 time
// steps: 3.98 ms with streaming chunks, 2.99 ms here.
#include "jacobi2d.hpp"

using namespace rpx;

namespace {

typedef double v2d __attribute__((ext_vector_type(2)));
typedef v2d v2d_u __attribute__((aligned(8)));  // rows of an odd N start on 8 bytes

constexpr int kTileCols = 128;

__device__ __forceinline__ double point(double c, double w, double e, double s, double n) {
  return 0.2 * ((((c + w) + e) + s) + n);
}
// lane l receives v from lane l-1 (0 for lane 0) / from lane l+1 (0 for lane 63).
__device__ __forceinline__ double from_west(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x138, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x138, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_east(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x130, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x130, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

struct BlockArgs {
  double* Aout;        // interior written: level 2*steps
  double* B;           // interior written when store_b: level 2*steps - 1; its boundary is read
  const double* Ain;   // interior read
  const double* Abnd;  // the A whose boundary holds
  int64_t N;
  int64_t steps;
  int own_c, own_r, strips, chunks, store_b;
};

// Which columns of a tile are the grid's: none, lane 0's x (west strip),
// lane 63's y (east strip), or any lane's either (a grid within one tile).
enum Side { kInner, kWest, kEast, kAny };

// One sweep: dst = point(src) on this wavefront's RW rows.
template <int W, int RW, int SIDE>
__device__ __forceinline__ void block_sweep(v2d (&dst)[RW], const v2d (&src)[RW], v2d (*edge)[2][kWave], int wave,
                                            int lane, int first, int last, bool x_keep, bool y_keep) {
  edge[wave][0][lane] = src[0];
  edge[wave][1][lane] = src[RW - 1];
  auto row = [&](int i, const v2d& up, const v2d& dn) {
    const bool out = SIDE == kAny && (i <= first || i >= last);
    const v2d c = src[i];
    const double w = from_west(c.y), e = from_east(c.x);
    const double x = point(c.x, w, c.y, dn.x, up.x), y = point(c.y, c.x, e, dn.y, up.y);
    dst[i].x = (SIDE == kWest || SIDE == kAny) && (x_keep || out) ? dst[i].x : x;
    dst[i].y = (SIDE == kEast || SIDE == kAny) && (y_keep || out) ? dst[i].y : y;
  };
  constexpr int kMid = (RW + 1) / 2;
#pragma unroll
  for (int i = 1; i < kMid; ++i) row(i, src[i - 1], src[i + 1]);
  __syncthreads();
  const v2d up = edge[wave > 0 ? wave - 1 : 0][1][lane];
  const v2d dn = edge[wave < W - 1 ? wave + 1 : wave][0][lane];
#pragma unroll
  for (int i = kMid; i < RW - 1; ++i) row(i, src[i - 1], src[i + 1]);
  if (SIDE == kAny || first < 0) row(0, up, src[1]);
  if (SIDE == kAny || last >= RW) row(RW - 1, src[RW - 2], dn);
}

// first, last: this wavefront's rows of the grid's first and last row; -1 or
// less and RW or more where it has none.
template <int W, int RW, int SIDE>
__device__ __forceinline__ void block_tile(const BlockArgs& g, v2d (*edge)[W][2][kWave], int64_t rbase, int64_t j0,
                                           int wave, int lane, int r_begin, int r_end, int c_begin, int c_end) {
  const int64_t N = g.N, row0 = rbase + wave * RW, jl = j0 + 2 * lane;
  const int first = row0 == 0 ? 0 : -1;
  const int last = SIDE == kAny ? int(N - 1 - row0) : row0 + RW == N ? RW - 1 : RW;
  v2d a[RW], b[RW];
  bool x_keep = false, y_keep = false;
  if constexpr (SIDE == kWest) x_keep = lane == 0;
  if constexpr (SIDE == kEast) y_keep = lane == kWave - 1;
  if constexpr (SIDE == kAny) {
    x_keep = jl == 0 || jl >= N - 1;
    y_keep = jl + 1 >= N - 1;
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int64_t at = (row0 + i) * N + jl;
      a[i] = b[i] = v2d{0.0, 0.0};
      if (row0 + i < N) {
        if (jl < N) a[i].x = g.Ain[at], b[i].x = g.B[at];
        if (jl + 1 < N) a[i].y = g.Ain[at + 1], b[i].y = g.B[at + 1];
      }
    }
  } else {
    const int64_t at = row0 * N + jl;
#pragma unroll
    for (int i = 0; i < RW; ++i) a[i] = *reinterpret_cast<const v2d_u*>(g.Ain + at + i * N);
    if (first == 0) {
      a[0] = *reinterpret_cast<const v2d_u*>(g.Abnd + at);
      b[0] = *reinterpret_cast<const v2d_u*>(g.B + at);
    }
    if (last == RW - 1) {
      a[RW - 1] = *reinterpret_cast<const v2d_u*>(g.Abnd + at + (RW - 1) * N);
      b[RW - 1] = *reinterpret_cast<const v2d_u*>(g.B + at + (RW - 1) * N);
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      if (x_keep) a[i].x = g.Abnd[at + i * N], b[i].x = g.B[at + i * N];
      if (y_keep) a[i].y = g.Abnd[at + i * N + 1], b[i].y = g.B[at + i * N + 1];
    }
  }
  for (int64_t t = 0; t < g.steps; ++t) {
    // Opaque to the optimiser, which otherwise unrolls the boundary tests into
    // copies of the loop and spills.
    int first_row = __builtin_amdgcn_readfirstlane(first), last_row = __builtin_amdgcn_readfirstlane(last);
    asm volatile("" : "+s"(first_row), "+s"(last_row));
    block_sweep<W, RW, SIDE>(b, a, edge[0], wave, lane, first_row, last_row, x_keep, y_keep);
    block_sweep<W, RW, SIDE>(a, b, edge[1], wave, lane, first_row, last_row, x_keep, y_keep);
  }
  const bool x_own = 2 * lane >= c_begin && 2 * lane < c_end;
  const bool y_own = 2 * lane + 1 >= c_begin && 2 * lane + 1 < c_end;
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int k = wave * RW + i;
    if (k < r_begin || k >= r_end) continue;
    const int64_t at = (row0 + i) * N + jl;
    if (x_own && y_own) {
      *reinterpret_cast<v2d_u*>(g.Aout + at) = a[i];
      if (g.store_b) *reinterpret_cast<v2d_u*>(g.B + at) = b[i];
    } else if (x_own) {
      g.Aout[at] = a[i].x;
      if (g.store_b) g.B[at] = b[i].x;
    } else if (y_own) {
      g.Aout[at + 1] = a[i].y;
      if (g.store_b) g.B[at + 1] = b[i].y;
    }
  }
}

template <int W, int RW>
__global__ __launch_bounds__(W* kWave, 4) void jacobi_block_kernel(const BlockArgs g) {
  __shared__ v2d edge[2][W][2][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const unsigned tile = xcd_major(blockIdx.x, gridDim.x);
  const int strip = int(tile % unsigned(g.strips)), chunk = int(tile / unsigned(g.strips));
  const int halo = 2 * int(g.steps);
  int64_t j0 = int64_t(strip) * g.own_c, rbase = int64_t(chunk) * g.own_r;
  int c_begin = strip == 0 ? 1 : halo, c_end = halo + g.own_c;
  int r_begin = chunk == 0 ? 1 : halo, r_end = halo + g.own_r;
  if (strip == g.strips - 1) {
    c_begin += int(j0 - (g.N - kTileCols));
    j0 = g.N - kTileCols;
    c_end = kTileCols - 1;
  }
  if (chunk == g.chunks - 1) {
    r_begin += int(rbase - (g.N - W * RW));
    rbase = g.N - W * RW;
    r_end = W * RW - 1;
  }
  if (strip == 0)
    block_tile<W, RW, kWest>(g, edge, rbase, j0, wave, lane, r_begin, r_end, c_begin, c_end);
  else if (strip == g.strips - 1)
    block_tile<W, RW, kEast>(g, edge, rbase, j0, wave, lane, r_begin, r_end, c_begin, c_end);
  else
    block_tile<W, RW, kInner>(g, edge, rbase, j0, wave, lane, r_begin, r_end, c_begin, c_end);
}

// A whole grid of N <= 128 in one workgroup's registers.
template <int W, int RW>
__global__ __launch_bounds__(W* kWave) void jacobi_grid_kernel(const BlockArgs g) {
  __shared__ v2d edge[2][W][2][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  block_tile<W, RW, kAny>(g, edge, 0, 0, wave, lane, 1, int(g.N - 1), 1, int(g.N - 1));
}

// Tiles: W wavefronts of RW rows.  Few rows leave small grids enough tiles
// for 256 CUs; many rows recompute less halo on large ones.
struct TileShape {
  int waves, rows;
};
constexpr TileShape kShapes[] = {{8, 4}, {8, 5}, {16, 4}, {16, 5}, {8, 10}, {8, 11}};

template <int W, int RW>
int launch_block(const BlockArgs& g, hipStream_t s) {
  jacobi_block_kernel<W, RW><<<dim3(unsigned(g.strips) * unsigned(g.chunks)), dim3(W * kWave), 0, s>>>(g);
  return launch_status();
}

// The tile counts of a launch; false where the shape does not fit.
bool layout(BlockArgs& g, const TileShape& t) {
  const int rows = t.waves * t.rows;
  g.own_c = int(kTileCols - 4 * g.steps);
  g.own_r = int(rows - 4 * g.steps);
  if (g.own_c <= 0 || g.own_r <= 0 || g.N < kTileCols || g.N < rows) return false;
  const int64_t strips = 1 + ceil_div(g.N - kTileCols, g.own_c), chunks = 1 + ceil_div(g.N - rows, g.own_r);
  if (strips * chunks > INT32_MAX) return false;
  g.strips = int(strips);
  g.chunks = int(chunks);
  return true;
}

// Time of a launch in microseconds, a fit to launches of all shapes and
// depths at N = 131 to 8192 (within about 15%): 4 us, and the larger of the
// sweeps' issue time and one read and write of the grid at 5 TB/s.  A sweep
// of a tile takes 0.03 us + 0.033 us per row and SIMD; beyond 256 tiles a CU
// runs several, and the last round is 0.4 full on average.
double launch_us(BlockArgs g, const TileShape& t) {
  if (!layout(g, t)) return 1e30;
  const double tiles = double(g.strips) * g.chunks / 256.0;
  const double sweep = 0.03 + 0.033 * t.waves * t.rows / 4;
  const double compute = (tiles <= 1 ? 1.0 : tiles + 0.4) * 2 * double(g.steps) * sweep;
  const double memory = 16e-6 * double(g.N) * double(g.N) / 5.0;
  return 4.0 + (compute > memory ? compute : memory);
}

int launch_shape(BlockArgs g, int shape, hipStream_t s) {
  if (!layout(g, kShapes[shape])) return RPX_ERR_UNSUPPORTED;
  switch (shape) {
    case 0: return launch_block<8, 4>(g, s);
    case 1: return launch_block<8, 5>(g, s);
    case 2: return launch_block<16, 4>(g, s);
    case 3: return launch_block<16, 5>(g, s);
    case 4: return launch_block<8, 10>(g, s);
    default: return launch_block<8, 11>(g, s);
  }
}

}  // namespace

namespace rpx {

int jacobi_one_tile(double* A, double* B, int64_t N, int64_t tsteps, hipStream_t s) {
  const BlockArgs g{A, B, A, A, N, tsteps, 0, 0, 1, 1, 1};
  if (N <= 64)
    jacobi_grid_kernel<16, 4><<<dim3(1), dim3(16 * kWave), 0, s>>>(g);
  else
    jacobi_grid_kernel<8, 16><<<dim3(1), dim3(8 * kWave), 0, s>>>(g);
  return launch_status();
}

// The plan: at least two launches (a launch never writes the grid it reads),
// their depths equal to within one, the shape and the number of launches of
// the least time.  An even number ping-pongs A -> Q -> A; an odd one begins
// A -> B -> Q, B's interior being free until the last launch stores it.
int jacobi_blocks(double* A, double* B, double* Q, int64_t N, int64_t tsteps, hipStream_t s) {
  double best = 1e30;
  int shape = -1;
  int64_t launches = 0;
  constexpr int64_t kMaxSteps = 14;
  for (int k = 0; k < int(sizeof(kShapes) / sizeof(kShapes[0])); ++k) {
    for (int64_t d = 1; d <= kMaxSteps && d < tsteps; ++d) {
      const int64_t n = ceil_div(tsteps, d) < 2 ? 2 : ceil_div(tsteps, d);
      BlockArgs g{};
      g.N = N;
      g.steps = tsteps / n;
      const int64_t deeper = tsteps % n;
      double us = double(n - deeper) * launch_us(g, kShapes[k]);
      ++g.steps;
      if (deeper > 0) us += double(deeper) * launch_us(g, kShapes[k]);
      if (us < best) best = us, shape = k, launches = n;
    }
  }
  if (shape < 0) return RPX_ERR_UNSUPPORTED;
  double* src = A;
  for (int64_t i = 0; i < launches; ++i) {
    const int64_t left = launches - i;
    double* dst = left % 2 == 1 ? A : Q;
    if (i == 0 && launches % 2 == 1) dst = B;
    const BlockArgs g{dst, B, src, A, N, tsteps / launches + (i < tsteps % launches), 0, 0, 0, 0, left == 1};
    const int rc = launch_shape(g, shape, s);
    if (rc != RPX_SUCCESS) return rc;
    src = dst;
  }
  return RPX_SUCCESS;
}

}  // namespace rpx
