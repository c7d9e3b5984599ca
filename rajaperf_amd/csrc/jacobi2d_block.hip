// JACOBI_2D, several time steps per launch on one register-resident tile per
// workgroup.
//
// Reference: src/polybench/POLYBENCH_JACOBI_2D-Seq.cpp:30-54 (tsteps x two
// sweeps over the interior).
//
// Two forms of tile.  In the narrow one a workgroup of W wavefronts holds W*RW
// rows of 128 columns: a lane holds
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
// steps: 3.98 ms with streaming chunks, 2.96 ms on narrow tiles of 88 rows,
// 2.61 ms on wide ones (below).
#include "jacobi2d.hpp"

#include <cmath>

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

// ---- wide tiles --------------------------------------------------------------
//
// 256 columns: a lane holds four columns of RW rows, once, and a sweep replaces
// them in place: half the registers per point, so twice the columns and less
// halo, and four DPP moves for 20 FP64 instructions instead of 10 (a row and
// sweep of 256 columns takes 127 clocks, two of 128 columns 128, but 61 of 100
// points of an 88-row tile are kept at seven steps, 51 of an 80-row narrow one).
// N = 8192, 50 steps: seven launches of seven or eight steps, about 370 us each,
// 165 of which the memory needs and about 310 the instructions, in part one
// after the other: two workgroups per CU are all that the registers hold.  From
// N = 2000 or so; smaller grids have too few of them.
// The grid's boundary cells, which the A and the B level have of their own,
// wait in LDS for the tiles that hold any.
constexpr int kWideCols = 256;

template <int W, int RW>
struct WideRoom {
  v2d edge[2][W][2][2][kWave];   // [parity][wavefront][first or last row][pair]
  v2d row[2][2][2][kWave];       // the grid's first or last row, [A or B][pair]
  double column[2][W * RW];      // its first or last column, [A or B]
};

typedef double Quad[4];
__device__ __forceinline__ void put_quad(v2d (*to)[kWave], int lane, const Quad& q) {
  to[0][lane] = v2d{q[0], q[1]};
  to[1][lane] = v2d{q[2], q[3]};
}
__device__ __forceinline__ void get_quad(Quad& q, const v2d (*from)[kWave], int lane) {
  const v2d l = from[0][lane], r = from[1][lane];
  q[0] = l.x, q[1] = l.y, q[2] = r.x, q[3] = r.y;
}
__device__ __forceinline__ void load_quad(Quad& q, const double* from) {
  const v2d l = *reinterpret_cast<const v2d_u*>(from), r = *reinterpret_cast<const v2d_u*>(from + 2);
  q[0] = l.x, q[1] = l.y, q[2] = r.x, q[3] = r.y;
}

// One sweep.  q[RW + 1] holds the A level's row i in q[i + 1] and the B level's
// in q[i]: the sweep from A to B (LEVEL = 1) goes down and puts each new row
// where the old row above it was, the sweep back goes up and puts it where the
// old row below it was.
template <int W, int RW, int SIDE, int LEVEL>
__device__ __forceinline__ void wide_sweep(Quad (&q)[RW + 1], WideRoom<W, RW>& m, int wave, int lane, bool first,
                                           bool last) {
  // Row i, with its old neighbours up and dn.
  auto row = [&](int i, const Quad& up, const Quad& dn) {
    const Quad& c = q[i + LEVEL];
    Quad r;
    const double w = from_west(c[3]), e = from_east(c[0]);
    r[0] = point(c[0], w, c[1], dn[0], up[0]);
    r[1] = point(c[1], c[0], c[2], dn[1], up[1]);
    r[2] = point(c[2], c[1], c[3], dn[2], up[2]);
    r[3] = point(c[3], c[2], e, dn[3], up[3]);
    if (SIDE == kWest) r[0] = lane == 0 ? m.column[LEVEL][wave * RW + i] : r[0];
    if (SIDE == kEast) r[3] = lane == kWave - 1 ? m.column[LEVEL][wave * RW + i] : r[3];
    // Pinned: the optimiser otherwise moves the rows' last steps behind the
    // branches below, old rows and all, and spills.
    asm volatile("" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]));
    __builtin_amdgcn_sched_barrier(0);  // one row at a time
#pragma unroll
    for (int k = 0; k < 4; ++k) q[i + 1 - LEVEL][k] = r[k];
  };
  auto top = [&] {
    if (first) {
      get_quad(q[1 - LEVEL], m.row[0][LEVEL], lane);
    } else {
      Quad up;
      get_quad(up, m.edge[1 - LEVEL][wave > 0 ? wave - 1 : 0][1], lane);
      row(0, up, q[1 + LEVEL]);
    }
    put_quad(m.edge[LEVEL][wave][0], lane, q[1 - LEVEL]);
  };
  auto bottom = [&] {
    if (last) {
      get_quad(q[RW - LEVEL], m.row[1][LEVEL], lane);
    } else {
      Quad dn;
      get_quad(dn, m.edge[1 - LEVEL][wave < W - 1 ? wave + 1 : wave][0], lane);
      row(RW - 1, q[RW - 2 + LEVEL], dn);
    }
    put_quad(m.edge[LEVEL][wave][1], lane, q[RW - LEVEL]);
  };
  if (LEVEL == 1) {
    top();
#pragma unroll
    for (int i = 1; i < RW - 1; ++i) row(i, q[i], q[i + 2]);
    bottom();
  } else {
    bottom();
#pragma unroll
    for (int i = RW - 2; i > 0; --i) row(i, q[i - 1], q[i + 1]);
    top();
  }
  __syncthreads();
}

// LAST: the launch that stores the last B as well.
template <int W, int RW, int SIDE, bool LAST>
__device__ __forceinline__ void wide_tile(const BlockArgs& g, WideRoom<W, RW>& m, int64_t rbase, int64_t j0, int wave,
                                          int lane, int r_begin, int r_end, int c_begin, int c_end) {
  const int64_t N = g.N, row0 = rbase + wave * RW, at0 = row0 * N + j0 + 4 * lane;
  const int first = row0 == 0, last = row0 + RW == N;
  Quad q[RW + 1];  // A's row i in q[i + 1]
#pragma unroll
  for (int i = 0; i < RW; ++i) load_quad(q[i + 1], g.Ain + at0 + i * N);
#pragma unroll
  for (int k = 0; k < 4; ++k) q[0][k] = 0.0;
  auto boundary_row = [&](Quad& r, int64_t at, v2d (*room)[2][kWave]) {
    load_quad(r, g.B + at);
    put_quad(room[1], lane, r);
    load_quad(r, g.Abnd + at);
    put_quad(room[0], lane, r);
  };
  if (first) boundary_row(q[1], at0, m.row[0]);
  if (last) boundary_row(q[RW], at0 + (RW - 1) * N, m.row[1]);
  if (SIDE != kInner) {
    const int64_t edge_col = SIDE == kWest ? 0 : N - 1;
    if (lane < RW) {
      m.column[0][wave * RW + lane] = g.Abnd[(row0 + lane) * N + edge_col];
      m.column[1][wave * RW + lane] = g.B[(row0 + lane) * N + edge_col];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const double b = m.column[0][wave * RW + i];
      if (SIDE == kWest) q[i + 1][0] = lane == 0 ? b : q[i + 1][0];
      else q[i + 1][3] = lane == kWave - 1 ? b : q[i + 1][3];
    }
  }
  put_quad(m.edge[0][wave][0], lane, q[1]);
  put_quad(m.edge[0][wave][1], lane, q[RW]);
  __syncthreads();
  auto store = [&](double* out, int slot) {
    int64_t base = at0;  // opaque, or the addresses of all rows are kept through the time steps
    asm volatile("" : "+v"(base));
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int k = wave * RW + i;
      if (k < r_begin || k >= r_end) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int c = 4 * lane + 2 * h;
        const bool x_own = c >= c_begin && c < c_end, y_own = c + 1 >= c_begin && c + 1 < c_end;
        double* at = out + base + i * N + 2 * h;
        if (x_own && y_own) *reinterpret_cast<v2d_u*>(at) = v2d{q[i + slot][2 * h], q[i + slot][2 * h + 1]};
        if (SIDE == kInner) continue;  // whole pairs
        if (x_own && !y_own) at[0] = q[i + slot][2 * h];
        if (y_own && !x_own) at[1] = q[i + slot][2 * h + 1];
      }
    }
  };
  // Opaque to the optimiser, which otherwise makes copies of the loop.
  int is_first, is_last;
  auto opaque = [&] {
    is_first = __builtin_amdgcn_readfirstlane(first), is_last = __builtin_amdgcn_readfirstlane(last);
    asm volatile("" : "+s"(is_first), "+s"(is_last));
  };
  for (int64_t t = LAST; t < g.steps; ++t) {
    opaque();
    wide_sweep<W, RW, SIDE, 1>(q, m, wave, lane, is_first, is_last);
    wide_sweep<W, RW, SIDE, 0>(q, m, wave, lane, is_first, is_last);
  }
  if (LAST) {
    opaque();
    wide_sweep<W, RW, SIDE, 1>(q, m, wave, lane, is_first, is_last);
    store(g.B, 0);
    wide_sweep<W, RW, SIDE, 0>(q, m, wave, lane, is_first, is_last);
  }
  store(g.Aout, 1);
}

template <int W, int RW, bool LAST>
__global__ __launch_bounds__(W* kWave, 4) void jacobi_wide_kernel(const BlockArgs g) {
  __shared__ WideRoom<W, RW> room;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const unsigned tile = xcd_major(blockIdx.x, gridDim.x);
  const int strip = int(tile % unsigned(g.strips)), chunk = int(tile / unsigned(g.strips));
  const int halo = 2 * int(g.steps);
  int64_t j0 = int64_t(strip) * g.own_c, rbase = int64_t(chunk) * g.own_r;
  int c_begin = strip == 0 ? 1 : halo, c_end = halo + g.own_c;
  int r_begin = chunk == 0 ? 1 : halo, r_end = halo + g.own_r;
  if (strip == g.strips - 1) {
    c_begin += int(j0 - (g.N - kWideCols));
    j0 = g.N - kWideCols;
    c_end = kWideCols - 1;
  }
  if (chunk == g.chunks - 1) {
    r_begin += int(rbase - (g.N - W * RW));
    rbase = g.N - W * RW;
    r_end = W * RW - 1;
  }
  if (strip == 0)
    wide_tile<W, RW, kWest, LAST>(g, room, rbase, j0, wave, lane, r_begin, r_end, c_begin, c_end);
  else if (strip == g.strips - 1)
    wide_tile<W, RW, kEast, LAST>(g, room, rbase, j0, wave, lane, r_begin, r_end, c_begin, c_end);
  else
    wide_tile<W, RW, kInner, LAST>(g, room, rbase, j0, wave, lane, r_begin, r_end, c_begin, c_end);
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
  int waves, rows, cols;
  double sweep_us;  // one sweep of a tile on a CU that has as many as it holds, per tile
  double tbps;      // rate of a launch of few steps, which the memory bounds
};
constexpr TileShape kShapes[] = {{8, 4, kTileCols, 0.23, 4.75},  {8, 5, kTileCols, 0.295, 4.7},
                                 {16, 4, kTileCols, 0.48, 4.65}, {16, 5, kTileCols, 0.78, 4.5},
                                 {8, 10, kWideCols, 1.05, 4.1},  {8, 11, kWideCols, 1.145, 4.1}};

template <int W, int RW>
int launch_wide(const BlockArgs& g, hipStream_t s) {
  const dim3 grid(unsigned(g.strips) * unsigned(g.chunks)), block(W * kWave);
  if (g.store_b) jacobi_wide_kernel<W, RW, true><<<grid, block, 0, s>>>(g);
  else jacobi_wide_kernel<W, RW, false><<<grid, block, 0, s>>>(g);
  return launch_status();
}

template <int W, int RW>
int launch_block(const BlockArgs& g, hipStream_t s) {
  jacobi_block_kernel<W, RW><<<dim3(unsigned(g.strips) * unsigned(g.chunks)), dim3(W * kWave), 0, s>>>(g);
  return launch_status();
}

// The tile counts of a launch; false where the shape does not fit.
bool layout(BlockArgs& g, const TileShape& t) {
  const int rows = t.waves * t.rows;
  g.own_c = int(t.cols - 4 * g.steps);
  g.own_r = int(rows - 4 * g.steps);
  if (g.own_c <= 0 || g.own_r <= 0 || g.N <= t.cols || g.N < rows) return false;
  const int64_t strips = 1 + ceil_div(g.N - t.cols, g.own_c), chunks = 1 + ceil_div(g.N - rows, g.own_r);
  if (strips * chunks > INT32_MAX) return false;
  g.strips = int(strips);
  g.chunks = int(chunks);
  return true;
}

// Time of a launch in microseconds, a fit to launches of all shapes and depths
// at 16 grids from N = 300 to 8192 (the shape and depth that it picks are
// within 3% of the fastest at all of them): 4.6 us, the sweeps' issue time, and
// one read and write of the grid (slowest with wide tiles, whose lanes read and
// write every other 16 bytes), which overlap in part.  A CU works on two
// tiles at a time; an odd one out is alone, and its wavefronts then wait for
// each other's edge rows.  Beyond four tiles per CU this evens out.
double launch_us(BlockArgs g, const TileShape& t) {
  if (!layout(g, t)) return 1e30;
  const bool wide = t.cols == kWideCols;
  const double tiles = double(g.strips) * g.chunks / 256.0, n = std::ceil(tiles), alone = wide ? 1.36 : 1.07;
  const double rounds = n > 4 ? tiles : std::fmod(n, 2.0) == 1.0 ? n - 1 + alone : n;
  const double sweeps = rounds * 2 * double(g.steps) * t.sweep_us;
  const double memory = 16e-6 * double(g.N) * double(g.N) / t.tbps;
  return 4.6 + std::cbrt(sweeps * sweeps * sweeps + memory * memory * memory);
}

int launch_shape(BlockArgs g, int shape, hipStream_t s) {
  if (!layout(g, kShapes[shape])) return RPX_ERR_UNSUPPORTED;
  switch (shape) {
    case 0: return launch_block<8, 4>(g, s);
    case 1: return launch_block<8, 5>(g, s);
    case 2: return launch_block<16, 4>(g, s);
    case 3: return launch_block<16, 5>(g, s);
    case 4: return launch_wide<8, 10>(g, s);
    default: return launch_wide<8, 11>(g, s);
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
