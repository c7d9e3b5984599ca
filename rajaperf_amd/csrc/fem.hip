// MASS3DPA and DIFFUSION3DPA: partial-assembly operator actions on hex
// elements, sum-factorised, FP64.
//
// Reference: src/apps/MASS3DPA.hpp:158-339 with MASS3DPA-Seq.cpp:29-94, and
// src/apps/DIFFUSION3DPA.hpp:216-458 with DIFFUSION3DPA-Seq.cpp:28-110.  The
// suite's HIP variants run one element per workgroup of (Q1D,Q1D[,Q1D])
// work-items with 8-9 barriers (MASS3DPA-Hip.cpp:25-111,
// DIFFUSION3DPA-Hip.cpp:25-134).
//
// MI355X design: a workgroup of 256 work-items owns E elements, as many as have
// a work-item for every pencil of the widest stage.  Each of the six
// contraction stages maps one work-item to one 1D "pencil" of one element
// (e.g. the x-contraction to the (e,dz,dy) pencils), keeps the pencil in
// registers and replaces it in LDS by its result; stages are separated by
// workgroup barriers, so a workgroup takes 5 barriers per E elements.  X and
// the quadrature data are read once with coalesced pencil loads, Y is
// updated in place, the basis tables come through the scalar cache.  The
// contraction order of every stage and the association of every sum are those
// of the Base_Seq loops and no multiply-add is fused, so results are
// bit-identical to Base_Seq.
//
// Stage order (forward x, y, z; backward x, y, z):
//   P1 (e,dz,dy): DDQ[dz][dy][qx] = sum_dx X[dz][dy][dx] B(qx,dx)
//   P2 (e,dz,qx): DQQ[dz][qy][qx] = sum_dy DDQ[dz][dy][qx] B(qy,dy)
//   P3 (e,qy,qx): QQQ[qz][qy][qx] = (sum_dz DQQ[dz][qy][qx] B(qz,dz)) * D
//   P4 (e,qz,qy): QQD[qz][qy][dx] = sum_qx QQQ[qz][qy][qx] Bt'(dx,qx)
//   P5 (e,qz,dx): QDD[qz][dy][dx] = sum_qy QQD[qz][qy][dx] Bt'(dy,qy)
//   P6 (e,dy,dx): Y[dz][dy][dx]  += sum_qz QDD[qz][dy][dx] Bt'(dz,qz)
// with B(q,d) = B[q + Q*d] and the suite's literal Bt'(d,q) = Bt[q + D*d]
// (MASS3DPA.hpp:175).  DIFFUSION3DPA carries three components per stage.
#include "rpx_common.hpp"
#include "fem_common.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

using namespace rpx;

namespace {

constexpr int kBS = 256;

// Global-memory pointers: with the address space in the type, accesses are
// global (not FLAT) instructions even where the pointer comes from memory.
typedef const __attribute__((address_space(1))) double gcdouble;
typedef __attribute__((address_space(1))) double gdouble;

// Basis tables are read through the scalar cache into SGPRs, which a multiply
// takes as its uniform operand: they cost no LDS bandwidth and no VGPRs.  (A
// broadcast LDS read of a basis value costs as much LDS time as one of 64
// different values; re-read per pencil they were 80% of the LDS traffic at
// (8,9).)  The pointer is made opaque where a stage begins, so that a table
// is loaded for one stage and not kept over all of them.
typedef const __attribute__((address_space(4))) double cdouble;
__device__ __forceinline__ cdouble* table(gcdouble* p) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(a));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(a >> 32));
  return reinterpret_cast<cdouble*>(uint64_t(hi) << 32 | lo);
}
__device__ __forceinline__ cdouble* opaque(cdouble* p) {
  asm volatile("" : "+s"(p));
  return p;
}
// u[q] = sum_d v[d] B(q,d), B(q,d) = T[q + Q*d].
template <int D, int Q>
__device__ __forceinline__ void to_quad(const double (&v)[D], cdouble* T, double (&u)[Q]) {
#pragma unroll
  for (int q = 0; q < Q; ++q) u[q] = 0.0;
#pragma unroll
  for (int d = 0; d < D; ++d)
#pragma unroll
    for (int q = 0; q < Q; ++q) u[q] += v[d] * T[q + Q * d];
}

// u[d] = sum_q v[q] Bt'(d,q), Bt'(d,q) = T[q + D*d].
template <int D, int Q>
__device__ __forceinline__ void to_dofs(const double (&v)[Q], cdouble* T, double (&u)[D]) {
#pragma unroll
  for (int d = 0; d < D; ++d) {
    u[d] = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) u[d] += v[q] * T[q + D * d];
  }
}

// E elements per workgroup, so that no stage has more pencils than there are
// work-items: the Q^2 of the widest stage fill them as far as they go.  What
// bounds the operator is then the memory it moves: at NE = 185185 / 116618 /
// 78125 of D1D = 6 / 7 / 8 it takes 264 / 260 / 269 us (0.80-0.85 of the time
// of its bytes at 6.5 TB/s).  With as many elements as 24 to 48 KB of LDS hold
// a stage took two passes, the second nearly empty, and fewer workgroups fit
// on a CU: 278 / 312 / 317 us; with the basis in LDS as well 324 / 396 / 388 us.
// (4,5) at NE = 600000: 281 us, 234 at 6.5 TB/s.
template <int D, int Q>
struct MassShape {
  static constexpr int Q3 = Q * Q * Q;  // doubles of LDS per element
  static constexpr int E = kBS / (Q * Q);
  static constexpr int kLds = E * Q3;
};

// Elements [e0, e0+ne) of one operator application, ne <= MassShape::E, by
// the whole workgroup, in an LDS grid [qz][qy][qx] per element: every stage
// reads and writes the same rows or columns of it, one work-item each, and
// only their lengths change.  Ends with the workgroup's last LDS reads still
// pending: a caller that reuses the buffer must synchronise first.
template <int D, int Q, bool kEarlyXY = true>
__device__ __forceinline__ void mass3dpa_elements(gcdouble* __restrict__ Bg, gcdouble* __restrict__ Btg,
                                                  gcdouble* __restrict__ Dg, gcdouble* __restrict__ Xg,
                                                  gdouble* __restrict__ Yg, int64_t e0, int ne,
                                                  double* __restrict__ buf) {
  constexpr int D2 = D * D, D3 = D * D * D, Q2 = Q * Q, Q3 = Q * Q * Q;
  const int w = threadIdx.x;  // the pencil of every stage
  cdouble* const Bc = table(Bg);
  cdouble* const Btc = table(Btg);

  // D (P3), X (P1) and Y (P6) pencils go to registers early: D and X before
  // P1, Y at the start of P4 (when D's registers are free), so none of these
  // loads waits at the head of its stage.  X and Y not at Q = D + 2 from D = 5
  // nor in the persistent loops (the single-launch batch kernel and the
  // per-order loop), where the extra live registers cost a wavefront per SIMD.
  constexpr bool kPreXY = kEarlyXY && !(D >= 5 && Q >= D + 2);
  gcdouble* const xp = Xg + (e0 + w / D2) * D3 + w % D2 * D;  // X[e][dz][dy][:]
  gdouble* const yp = Yg + (e0 + w / D2) * D3 + w % D2;       // Y[e][:][dy][dx]
  double x[D], y[D], dq[Q];
  auto load_x = [&] {
#pragma unroll
    for (int dx = 0; dx < D; ++dx) x[dx] = xp[dx];
  };
  // All of the pencil's Y values are loaded before the first store: where the
  // Y pointer comes from memory the compiler otherwise keeps each load behind
  // the previous store and waits on it D times per pencil.
  auto load_y = [&] {
#pragma unroll
    for (int dz = 0; dz < D; ++dz) y[dz] = yp[dz * D2];
  };
  if (kPreXY && w < ne * D2) load_x();
  if (w < ne * Q2) {
    gcdouble* dp = Dg + (e0 + w / Q2) * Q3 + w % Q2;
#pragma unroll
    for (int qz = 0; qz < Q; ++qz) dq[qz] = dp[qz * Q2];
  }

  // P1: x-contraction of X pencils, to row dy of plane dz.
  cdouble* T = opaque(Bc);
  if (w < ne * D2) {
    if constexpr (!kPreXY) load_x();
    double u[Q];
    to_quad<D, Q>(x, T, u);
    double* out = buf + w / D2 * Q3 + w % D2 / D * Q2 + w % D * Q;
#pragma unroll
    for (int qx = 0; qx < Q; ++qx) out[qx] = u[qx];
  }
  __syncthreads();
  // P2: y-contraction, column qx of plane dz.
  T = opaque(Bc);
  if (w < ne * D * Q) {
    const int e = w / (D * Q), r = w % (D * Q);
    double* col = buf + e * Q3 + r / Q * Q2 + r % Q;
    double v[D], u[Q];
#pragma unroll
    for (int dy = 0; dy < D; ++dy) v[dy] = col[dy * Q];
    to_quad<D, Q>(v, T, u);
#pragma unroll
    for (int qy = 0; qy < Q; ++qy) col[qy * Q] = u[qy];
  }
  __syncthreads();
  // P3: z-contraction and the quadrature-point scaling, column (qy, qx).
  T = opaque(Bc);
  if (w < ne * Q2) {
    double* col = buf + w / Q2 * Q3 + w % Q2;
    double v[D], u[Q];
#pragma unroll
    for (int dz = 0; dz < D; ++dz) v[dz] = col[dz * Q2];
    to_quad<D, Q>(v, T, u);
#pragma unroll
    for (int qz = 0; qz < Q; ++qz) col[qz * Q2] = u[qz] * dq[qz];
  }
  __syncthreads();
  if (kPreXY && w < ne * D2) load_y();
  // P4: backward x-contraction, row (qz, qy).
  T = opaque(Btc);
  if (w < ne * Q2) {
    double* row = buf + w * Q;
    double v[Q], u[D];
#pragma unroll
    for (int qx = 0; qx < Q; ++qx) v[qx] = row[qx];
    to_dofs<D, Q>(v, T, u);
#pragma unroll
    for (int dx = 0; dx < D; ++dx) row[dx] = u[dx];
  }
  __syncthreads();
  // P5: backward y-contraction, column dx of plane qz.
  T = opaque(Btc);
  if (w < ne * Q * D) {
    const int e = w / (Q * D), r = w % (Q * D);
    double* col = buf + e * Q3 + r / D * Q2 + r % D;
    double v[Q], u[D];
#pragma unroll
    for (int qy = 0; qy < Q; ++qy) v[qy] = col[qy * Q];
    to_dofs<D, Q>(v, T, u);
#pragma unroll
    for (int dy = 0; dy < D; ++dy) col[dy * Q] = u[dy];
  }
  __syncthreads();
  // P6: backward z-contraction of column (dy, dx), accumulate into Y.
  T = opaque(Btc);
  if (w < ne * D2) {
    const double* col = buf + w / D2 * Q3 + w % D2 / D * Q + w % D;
    double v[Q], u[D];
#pragma unroll
    for (int qz = 0; qz < Q; ++qz) v[qz] = col[qz * Q2];
    if constexpr (!kPreXY) load_y();
    to_dofs<D, Q>(v, T, u);
#pragma unroll
    for (int dz = 0; dz < D; ++dz) yp[dz * D2] = y[dz] + u[dz];
  }
}

template <int D, int Q>
__global__ __launch_bounds__(kBS) void mass3dpa_kernel(const double* __restrict__ Bg,
                                                       const double* __restrict__ Btg,
                                                       const double* __restrict__ Dg,
                                                       const double* __restrict__ Xg, double* __restrict__ Yg,
                                                       int64_t NE) {
  using S = MassShape<D, Q>;
  __shared__ double buf[S::kLds];
  const int64_t e0 = int64_t(blockIdx.x) * S::E;
  const int ne = int((NE - e0) < S::E ? (NE - e0) : S::E);
  mass3dpa_elements<D, Q>((gcdouble*)Bg, (gcdouble*)Btg, (gcdouble*)Dg, (gcdouble*)Xg, (gdouble*)Yg, e0, ne, buf);
}

// ---- ragged batches, one persistent launch ----------------------------------
//
// A batch is one operator application (its own bases, data and order, with
// Q1D = D1D + 1).  Batch b is cut into chunks of MassShape<D,Q>::E elements;
// chunk c belongs to batch chunk_batch[c], whose first chunk is
// chunk0[batch].  A grid of a few workgroups per CU strides over the chunks;
// each chunk dispatches on its batch's order to the same element code as the
// single-order kernel, so results are bit-identical to it.
// Doubles: the largest kLds over the orders.
constexpr int kBatchLds = MassShape<8, 9>::kLds > MassShape<7, 8>::kLds ? MassShape<8, 9>::kLds : MassShape<7, 8>::kLds;

typedef __attribute__((address_space(3))) double lds_double;

// One chunk of a batch of order D.  Not inlined: each order's element code
// keeps its own register allocation.  The LDS pointer keeps its address space
// across the call so its accesses stay LDS instructions.  64 batches of orders
// 2..8 (1.08 M elements): 1.57 ms in this one launch, 1.52 with a
// single-order launch per batch and 1.28 with a launch per order
// (mass3dpa_order_chunk_kernel), the default.
template <int D>
__device__ __attribute__((noinline)) void mass_batch_chunk(rpx_mass_batch b, int64_t e0, lds_double* lds) {
  using S = MassShape<D, D + 1>;
  static_assert(S::kLds <= kBatchLds, "LDS budget");
  const int ne = int((b.ne - e0) < S::E ? (b.ne - e0) : S::E);
  // The descriptors' pointers are global memory: typed so, the element code
  // issues global (not FLAT) accesses, which do not hold up its LDS waits.
  mass3dpa_elements<D, D + 1, false>((gcdouble*)b.B, (gcdouble*)b.Bt, (gcdouble*)b.D, (gcdouble*)b.X, (gdouble*)b.Y, e0, ne,
                                    (double*)lds);
}

// Elements per chunk of a batch of order d1d (Q1D = d1d + 1).
__host__ __device__ inline int64_t batch_chunk_elems(int d1d) {
  switch (d1d) {
    case 1: return MassShape<1, 2>::E;
    case 2: return MassShape<2, 3>::E;
    case 3: return MassShape<3, 4>::E;
    case 4: return MassShape<4, 5>::E;
    case 5: return MassShape<5, 6>::E;
    case 6: return MassShape<6, 7>::E;
    case 7: return MassShape<7, 8>::E;
    default: return MassShape<8, 9>::E;
  }
}

// Scratch of a batched plan: a 256-byte header (the chunk count), the batch
// descriptors, each chunk's batch, each batch's first chunk.
struct BatchHeader {
  int64_t nchunks;
  int64_t nbatch;
  int64_t order_begin[9];  // chunks of order d1d are [order_begin[d1d], order_end[d1d])
  int64_t order_end[9];
};
static_assert(sizeof(BatchHeader) <= 256, "plan header");

__host__ __device__ inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }
__host__ __device__ inline size_t chunk_batch_offset(int64_t nbatch) {
  return 256 + align256(size_t(nbatch) * sizeof(rpx_mass_batch));
}
__host__ __device__ inline size_t chunk0_offset(int64_t nbatch, int64_t nchunks) {
  return chunk_batch_offset(nbatch) + align256(size_t(nchunks) * sizeof(int));
}

// Chunks already run, per order: the first done[d] chunks of order d.
struct ChunkSkip {
  int64_t done[9];
};

// Every order's chunks after its first skip.done[d] (all of them for a zero
// skip), highest order first; plan order puts the orders' ranges in that
// order, so c only grows.
__global__ __launch_bounds__(kBS, 3) void mass3dpa_batched_kernel(const char* __restrict__ plan, ChunkSkip skip) {
  __shared__ double lds[kBatchLds];
  const BatchHeader* hdr = reinterpret_cast<const BatchHeader*>(plan);
  const int64_t nchunks = hdr->nchunks, nbatch = hdr->nbatch;
  const auto* batches = reinterpret_cast<const rpx_mass_batch*>(plan + 256);
  const auto* chunk_batch = reinterpret_cast<const int*>(plan + chunk_batch_offset(nbatch));
  const auto* chunk0 = reinterpret_cast<const int64_t*>(plan + chunk0_offset(nbatch, nchunks));
  rpx_mass_batch b{};
  int64_t cb = 0, ce = 0;  // chunk range of the batch held in b
  for (int d = 8; d >= 1; --d)
  for (int64_t c = hdr->order_begin[d] + skip.done[d] + blockIdx.x; c < hdr->order_end[d]; c += gridDim.x) {
    if (c >= ce) {  // the stride left b's chunks (each batch's are contiguous)
      const int bi = chunk_batch[c];
      b = batches[bi];
      cb = chunk0[bi];
      ce = cb + ceil_div(b.ne, batch_chunk_elems(b.d1d));
    }
    const int64_t k = c - cb;
    lds_double* l = (lds_double*)lds;
    switch (b.d1d) {
      case 1: mass_batch_chunk<1>(b, k * MassShape<1, 2>::E, l); break;
      case 2: mass_batch_chunk<2>(b, k * MassShape<2, 3>::E, l); break;
      case 3: mass_batch_chunk<3>(b, k * MassShape<3, 4>::E, l); break;
      case 4: mass_batch_chunk<4>(b, k * MassShape<4, 5>::E, l); break;
      case 5: mass_batch_chunk<5>(b, k * MassShape<5, 6>::E, l); break;
      case 6: mass_batch_chunk<6>(b, k * MassShape<6, 7>::E, l); break;
      case 7: mass_batch_chunk<7>(b, k * MassShape<7, 8>::E, l); break;
      default: mass_batch_chunk<8>(b, k * MassShape<8, 9>::E, l); break;
    }
    __syncthreads();  // the next chunk rewrites the LDS
  }
}

// The batches of one order, as one persistent launch over that order's range
// of the chunk table (the plan sorts batches by order, so the range is
// contiguous).  Same element code, LDS sizes and register allocation as the
// single-order kernel; an order with no batches exits at once.
template <int D>
__global__ __launch_bounds__(kBS) void mass3dpa_order_kernel(const char* __restrict__ plan) {
  using S = MassShape<D, D + 1>;
  __shared__ double buf[S::kLds];
  const BatchHeader* hdr = reinterpret_cast<const BatchHeader*>(plan);
  const int64_t nchunks = hdr->nchunks, nbatch = hdr->nbatch;
  const int64_t begin = hdr->order_begin[D], end = hdr->order_end[D];
  const auto* batches = reinterpret_cast<const rpx_mass_batch*>(plan + 256);
  const auto* chunk_batch = reinterpret_cast<const int*>(plan + chunk_batch_offset(nbatch));
  const auto* chunk0 = reinterpret_cast<const int64_t*>(plan + chunk0_offset(nbatch, nchunks));
  // Each batch's chunks are contiguous and c only grows, so the batch
  // descriptor is looked up again only when the stride leaves its range: a
  // lookup is a chain of three dependent loads, about 1-2 us, against a few
  // microseconds of work per chunk at the high orders.
  rpx_mass_batch b{};
  int64_t cb = 0, ce = 0;  // chunk range of the batch held in b
  for (int64_t c = begin + blockIdx.x; c < end; c += gridDim.x) {
    if (c >= ce) {
      const int bi = chunk_batch[c];
      b = batches[bi];
      cb = chunk0[bi];
      ce = cb + ceil_div(b.ne, int64_t(S::E));
    }
    const int64_t e0 = (c - cb) * S::E;
    const int ne = int((b.ne - e0) < S::E ? (b.ne - e0) : S::E);
    mass3dpa_elements<D, D + 1, false>((gcdouble*)b.B, (gcdouble*)b.Bt, (gcdouble*)b.D, (gcdouble*)b.X, (gdouble*)b.Y, e0,
                                ne, buf);
    __syncthreads();  // the next chunk rewrites the LDS
  }
}

// The batches of one order with one workgroup per chunk, for a grid of the
// order's chunk count.  Without the persistent loop around it the element
// code compiles as in the single-order kernel (at D1D = 8 62 VGPRs against 126,
// eight wavefronts per SIMD against four), and a chunk does not wait for the
// LDS reads of the one before: 64 batches of D1D = 7 / 8 (0.70 M elements) 1.60
// / 2.42 ms, 1.80 / 2.66 in the loop on 1024 workgroups.
template <int D>
__global__ __launch_bounds__(kBS) void mass3dpa_order_chunk_kernel(const char* __restrict__ plan) {
  using S = MassShape<D, D + 1>;
  __shared__ double buf[S::kLds];
  const BatchHeader* hdr = reinterpret_cast<const BatchHeader*>(plan);
  const int64_t nchunks = hdr->nchunks, nbatch = hdr->nbatch;
  const int64_t c = hdr->order_begin[D] + blockIdx.x;
  if (c >= hdr->order_end[D]) return;
  const auto* batches = reinterpret_cast<const rpx_mass_batch*>(plan + 256);
  const auto* chunk_batch = reinterpret_cast<const int*>(plan + chunk_batch_offset(nbatch));
  const auto* chunk0 = reinterpret_cast<const int64_t*>(plan + chunk0_offset(nbatch, nchunks));
  const int bi = chunk_batch[c];
  const rpx_mass_batch b = batches[bi];
  const int64_t e0 = (c - chunk0[bi]) * S::E;
  const int ne = int((b.ne - e0) < S::E ? (b.ne - e0) : S::E);
  mass3dpa_elements<D, D + 1>((gcdouble*)b.B, (gcdouble*)b.Bt, (gcdouble*)b.D, (gcdouble*)b.X, (gdouble*)b.Y, e0,
                              ne, buf);
}

template <int D>
int launch_order_chunks(const char* plan, int64_t chunks, hipStream_t s) {
  if (chunks <= 0) return RPX_SUCCESS;
  if (chunks > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  mass3dpa_order_chunk_kernel<D><<<dim3(unsigned(chunks)), dim3(kBS), 0, s>>>(plan);
  return launch_status();
}

// Chunk counts per order of the plans written by rpx_mass3dpa_batched_plan,
// kept on the host by scratch address so that a run sizes its grids without
// reading the device.  At most kMaxPlanRecords are kept (oldest dropped); a
// scratch without a record runs on the persistent kernels.
struct PlanRecord {
  const void* scratch;
  int64_t chunks[9];
};
constexpr size_t kMaxPlanRecords = 64;
std::mutex g_plan_mu;
std::vector<PlanRecord> g_plans;

void forget_plan(const void* scratch) {
  std::lock_guard<std::mutex> lock(g_plan_mu);
  g_plans.erase(std::remove_if(g_plans.begin(), g_plans.end(),
                               [&](const PlanRecord& r) { return r.scratch == scratch; }),
                g_plans.end());
}

void record_plan(const void* scratch, const int64_t* chunks) {
  std::lock_guard<std::mutex> lock(g_plan_mu);
  g_plans.erase(std::remove_if(g_plans.begin(), g_plans.end(),
                               [&](const PlanRecord& r) { return r.scratch == scratch; }),
                g_plans.end());
  if (g_plans.size() >= kMaxPlanRecords) g_plans.erase(g_plans.begin());
  PlanRecord r;
  r.scratch = scratch;
  std::copy(chunks, chunks + 9, r.chunks);
  g_plans.push_back(r);
}

bool find_plan(const void* scratch, int64_t* chunks) {
  std::lock_guard<std::mutex> lock(g_plan_mu);
  for (const PlanRecord& r : g_plans)
    if (r.scratch == scratch) {
      std::copy(r.chunks, r.chunks + 9, chunks);
      return true;
    }
  return false;
}

// Workgroups of mass3dpa_order_kernel<D> resident per CU (queried once).
template <int D>
int order_blocks_per_cu() {
  static int cached = 0;
  if (cached == 0) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, mass3dpa_order_kernel<D>, kBS, 0) != hipSuccess || n < 1)
      n = 1;
    cached = n;
  }
  return cached;
}

template <int D>
int launch_order(const char* plan, int cus, int64_t grid_override, hipStream_t s) {
  const int64_t grid = grid_override > 0 ? grid_override : int64_t(order_blocks_per_cu<D>()) * cus;
  if (grid > INT32_MAX) return RPX_ERR_INVALID_ARGUMENT;
  mass3dpa_order_kernel<D><<<dim3(unsigned(grid)), dim3(kBS), 0, s>>>(plan);
  return launch_status();
}

struct BatchLayout {
  int64_t nchunks;
  size_t batches_off, chunk_batch_off, chunk0_off, total;
};
BatchLayout batch_layout(const rpx_mass_batch* batches, int nbatch) {
  BatchLayout l;
  l.nchunks = 0;
  for (int i = 0; i < nbatch; ++i) l.nchunks += ceil_div(batches[i].ne, batch_chunk_elems(batches[i].d1d));
  l.batches_off = 256;
  l.chunk_batch_off = chunk_batch_offset(nbatch);
  l.chunk0_off = chunk0_offset(nbatch, l.nchunks);
  l.total = l.chunk0_off + align256(size_t(nbatch + 1) * sizeof(int64_t));
  return l;
}

// The plain FP64 comparator in the shape of the suite's Base_HIP variant
// (MASS3DPA-Hip.cpp:25-117): one element per workgroup of Q x Q work-items,
// two Q^3 LDS buffers, a barrier between stages.  Same sums in the same order
// as mass3dpa_kernel, so both are bit-identical to Base_Seq.
template <int D, int Q>
__global__ __launch_bounds__(Q* Q) void mass3dpa_naive_kernel(const double* __restrict__ Bg,
                                                               const double* __restrict__ Btg,
                                                               const double* __restrict__ Dg,
                                                               const double* __restrict__ Xg,
                                                               double* __restrict__ Yg) {
  constexpr int D2 = D * D, D3 = D * D * D, Q3 = Q * Q * Q;
  __shared__ double sB[Q * D];   // sB[q*D + d]  = B(q,d)
  __shared__ double sBt[D * Q];  // sBt[d*Q + q] = Bt'(d,q)
  __shared__ double s0[Q3];
  __shared__ double s1[Q3];
  const int tx = threadIdx.x % Q, ty = threadIdx.x / Q;
  const int64_t e = blockIdx.x;
  for (int t = threadIdx.x; t < Q * D; t += Q * Q) {
    sB[t] = Bg[t / D + Q * (t % D)];
    sBt[t] = Btg[t % Q + D * (t / Q)];
  }
  // X[dz][dy][dx] -> s0
  if (tx < D && ty < D)
    for (int dz = 0; dz < D; ++dz) s0[(dz * D + ty) * D + tx] = Xg[e * D3 + dz * D2 + ty * D + tx];
  __syncthreads();
  // x: s1[dz][dy][qx]   (tx = qx, ty = dy)
  if (ty < D)
    for (int dz = 0; dz < D; ++dz) {
      double u = 0.0;
      for (int dx = 0; dx < D; ++dx) u += s0[(dz * D + ty) * D + dx] * sB[tx * D + dx];
      s1[(dz * D + ty) * Q + tx] = u;
    }
  __syncthreads();
  // y: s0[dz][qy][qx]   (tx = qx, ty = qy)
  for (int dz = 0; dz < D; ++dz) {
    double u = 0.0;
    for (int dy = 0; dy < D; ++dy) u += s1[(dz * D + dy) * Q + tx] * sB[ty * D + dy];
    s0[(dz * Q + ty) * Q + tx] = u;
  }
  __syncthreads();
  // z and D: s1[qz][qy][qx]
  for (int qz = 0; qz < Q; ++qz) {
    double u = 0.0;
    for (int dz = 0; dz < D; ++dz) u += s0[(dz * Q + ty) * Q + tx] * sB[qz * D + dz];
    s1[(qz * Q + ty) * Q + tx] = u * Dg[e * Q3 + (qz * Q + ty) * Q + tx];
  }
  __syncthreads();
  // backward x: s0[qz][qy][dx]   (tx = dx, ty = qy)
  if (tx < D)
    for (int qz = 0; qz < Q; ++qz) {
      double u = 0.0;
      for (int qx = 0; qx < Q; ++qx) u += s1[(qz * Q + ty) * Q + qx] * sBt[tx * Q + qx];
      s0[(qz * Q + ty) * D + tx] = u;
    }
  __syncthreads();
  // backward y: s1[qz][dy][dx]   (tx = dx, ty = dy)
  if (tx < D && ty < D)
    for (int qz = 0; qz < Q; ++qz) {
      double u = 0.0;
      for (int qy = 0; qy < Q; ++qy) u += s0[(qz * Q + qy) * D + tx] * sBt[ty * Q + qy];
      s1[(qz * D + ty) * D + tx] = u;
    }
  __syncthreads();
  // backward z: Y[dz][dy][dx] +=
  if (tx < D && ty < D)
    for (int dz = 0; dz < D; ++dz) {
      double u = 0.0;
      for (int qz = 0; qz < Q; ++qz) u += s1[(qz * D + ty) * D + tx] * sBt[dz * Q + qz];
      Yg[e * D3 + dz * D2 + ty * D + tx] += u;
    }
}

// ---- DIFFUSION3DPA ----------------------------------------------------------

// Compile-time form of diffusion_tables: where in b or g the effective B(q,d)
// or G(q,d) sits, and G's sign.
template <int D, int Q>
struct HalfTables {
  static constexpr int key(int q, int d) { return d * Q + q; }
  static constexpr int sgn(int q, int d) { return q <= d ? -1 : 1; }
  static constexpr int b_at(int q, int d) {
    const int i = q <= d ? q : Q - 1 - q, j = q <= d ? d : D - 1 - d;
    const int mi = Q - 1 - i, mj = D - 1 - j;
    return key(i, j) > key(mi, mj) ? i + Q * j : mi + Q * mj;
  }
  static constexpr int g_at(int q, int d) {
    const int k = q <= d ? Q - 1 - q : q, l = q <= d ? D - 1 - d : d;
    const int nk = Q - 1 - k, nl = D - 1 - l;
    return key(k, l) > key(nk, nl) ? k + Q * l : nk + Q * nl;
  }
  static constexpr int g_sign(int q, int d) {
    const int k = q <= d ? Q - 1 - q : q, l = q <= d ? D - 1 - d : d;
    const int nk = Q - 1 - k, nl = D - 1 - l;
    return (key(k, l) > key(nk, nl) ? sgn(k, l) : sgn(nk, nl)) * sgn(q, d);
  }
  cdouble* b;
  cdouble* g;
  __device__ __forceinline__ double B(int q, int d) const { return b[b_at(q, d)]; }
  __device__ __forceinline__ double G(int q, int d) const { return g_sign(q, d) < 0 ? -g[g_at(q, d)] : g[g_at(q, d)]; }
  __device__ __forceinline__ HalfTables fresh() const { return {opaque(b), opaque(g)}; }
};

// The stages of the head of this file for three components, in one LDS grid of
// Q^3 per element and component: every stage reads and writes the same rows
// or columns of it, one work-item each, and only their lengths change, so no
// second buffer is needed and E elements fill the workgroup's lanes (as in
// MassShape).  What bounds it is the memory it moves, six tensor components
// per point: NE = 200000 of (4,5) takes 263 us, 232 at 6.5 TB/s; with two
// buffers, as many elements as 48 KB held and the basis in LDS it took 317.
// (8,9), NE = 26041: 317 us against 907.
template <int D, int Q, bool SYMM>
__global__ __launch_bounds__(kBS) void diffusion3dpa_kernel(const double* __restrict__ Bg,
                                                            const double* __restrict__ Gg,
                                                            const double* __restrict__ Dg,
                                                            const double* __restrict__ Xg,
                                                            double* __restrict__ Yg, int64_t NE) {
  constexpr int E = kBS / (Q * Q);
  constexpr int D2 = D * D, D3 = D * D * D, Q2 = Q * Q, Q3 = Q * Q * Q;
  constexpr int NC = SYMM ? 6 : 9;
  constexpr int K = 3 * Q3;  // doubles of an element; a component's stage result takes Q3 of them
  __shared__ double buf[E * K];
  const HalfTables<D, Q> tables{table((gcdouble*)Bg), table((gcdouble*)Gg)};

  const int w = threadIdx.x;  // the pencil of every stage
  const int64_t e0 = int64_t(blockIdx.x) * E;
  const int ne = int((NE - e0) < E ? (NE - e0) : E);
  const bool in1 = w < ne * D2, in2 = w < ne * D * Q, in3 = w < ne * Q2;

  // The point's tensor is loaded before P1 where it fits in the registers: (6,7)
  // 298 -> 258 us at NE = 61728; (8,9) 317 -> 332 at NE = 26041.
  constexpr bool kPreD = SYMM && Q <= 7;
  // From D1D = 7 the tables overflow the SGPRs; they are then re-read per row.
  constexpr bool kPerRow = D >= 7;
  double x[D], y[D], o[kPreD ? 6 : 1][Q];
  const double* const dp = Dg + (e0 + w / Q2) * (NC * Q3) + w % Q2;
  if (in1) {
    const double* xp = Xg + (e0 + w / D2) * D3 + w % D2 * D;
#pragma unroll
    for (int dx = 0; dx < D; ++dx) x[dx] = xp[dx];
  }
  if (kPreD && in3) {
#pragma unroll
    for (int c = 0; c < (kPreD ? 6 : 1); ++c)
#pragma unroll
      for (int qz = 0; qz < Q; ++qz) o[c][qz] = dp[c * Q3 + qz * Q2];
  }

  // P1 (DIFFUSION3DPA_3): DDQ0 = sum X*B, DDQ1 = sum X*G over dx.
  if (in1) {
    auto T = tables.fresh();
    double u[Q], v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) u[q] = v[q] = 0.0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (kPerRow) T = tables.fresh();
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        u[q] += x[d] * T.B(q, d);
        v[q] += x[d] * T.G(q, d);
      }
    }
    double* out = buf + w / D2 * K + w % D2 / D * Q2 + w % D * Q;  // rows dy of plane dz
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      out[q] = u[q];
      out[Q3 + q] = v[q];
    }
  }
  __syncthreads();
  // P2 (DIFFUSION3DPA_4): DQQ0 = sum DDQ1*B, DQQ1 = sum DDQ0*G, DQQ2 = sum DDQ0*B over dy.
  if (in2) {
    const int e = w / (D * Q), r = w % (D * Q);
    double* col = buf + e * K + r / Q * Q2 + r % Q;  // column qx of plane dz
    double a0[D], a1[D], u[Q], v[Q], t[Q];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      a0[d] = col[d * Q];
      a1[d] = col[Q3 + d * Q];
    }
    auto T = tables.fresh();
#pragma unroll
    for (int q = 0; q < Q; ++q) u[q] = v[q] = t[q] = 0.0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (kPerRow) T = tables.fresh();
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        u[q] += a1[d] * T.B(q, d);
        v[q] += a0[d] * T.G(q, d);
        t[q] += a0[d] * T.B(q, d);
      }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      col[q * Q] = u[q];
      col[Q3 + q * Q] = v[q];
      col[2 * Q3 + q * Q] = t[q];
    }
  }
  __syncthreads();
  // P3 (DIFFUSION3DPA_5): gradient at the point, times the symmetric tensor.
  if (in3) {
    double* col = buf + w / Q2 * K + w % Q2;
    double c0[D], c1[D], c2[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      c0[d] = col[d * Q2];
      c1[d] = col[Q3 + d * Q2];
      c2[d] = col[2 * Q3 + d * Q2];
    }
    auto T = tables.fresh();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (kPerRow) T = tables.fresh();
      double u = 0.0, v = 0.0, t = 0.0;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        u += c0[d] * T.B(q, d);
        v += c1[d] * T.B(q, d);
        t += c2[d] * T.G(q, d);
      }
      const double* op = dp + q * Q2;
      // Symmetric storage order (11, 12, 13, 22, 23, 33), DIFFUSION3DPA.hpp:384-392.
      const double O11 = kPreD ? o[0][q] : op[0];
      const double O12 = kPreD ? o[kPreD ? 1 : 0][q] : op[Q3];
      const double O13 = kPreD ? o[kPreD ? 2 : 0][q] : op[2 * Q3];
      const double O21 = SYMM ? O12 : op[3 * Q3];
      const double O22 = kPreD ? o[kPreD ? 3 : 0][q] : (SYMM ? op[3 * Q3] : op[4 * Q3]);
      const double O23 = kPreD ? o[kPreD ? 4 : 0][q] : (SYMM ? op[4 * Q3] : op[5 * Q3]);
      const double O31 = SYMM ? O13 : op[6 * Q3];
      const double O32 = SYMM ? O23 : op[7 * Q3];
      const double O33 = kPreD ? o[kPreD ? 5 : 0][q] : (SYMM ? op[5 * Q3] : op[8 * Q3]);
      col[q * Q2] = ((O11 * u) + (O12 * v)) + (O13 * t);
      col[Q3 + q * Q2] = ((O21 * u) + (O22 * v)) + (O23 * t);
      col[2 * Q3 + q * Q2] = ((O31 * u) + (O32 * v)) + (O33 * t);
    }
  }
  __syncthreads();
  double* const yp = Yg + (e0 + w / D2) * D3 + w % D2;
  if (in1) {
#pragma unroll
    for (int dz = 0; dz < D; ++dz) y[dz] = yp[dz * D2];
  }
  // Backward stages: component c's pencil times G where c == gc, B elsewhere.
  auto back = [&](const double* in, int stride, int gc, double (&u)[3][D]) {
    double c[3][Q];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int q = 0; q < Q; ++q) c[k][q] = in[k * Q3 + q * stride];
    auto T = tables.fresh();
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (kPerRow) T = tables.fresh();
      u[0][d] = u[1][d] = u[2][d] = 0.0;
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < 3; ++k) u[k][d] += c[k][q] * (k == gc ? T.G(q, d) : T.B(q, d));
    }
  };
  double u[3][D];
  // P4 (DIFFUSION3DPA_7): QQD0 = sum QQQ0*Gt, QQD1 = sum QQQ1*Bt, QQD2 = sum QQQ2*Bt
  // over qx, row r = qz*Q + qy.
  if (in3) {
    double* row = buf + w / Q2 * K + w % Q2 * Q;
    back(row, 1, 0, u);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int d = 0; d < D; ++d) row[k * Q3 + d] = u[k][d];
  }
  __syncthreads();
  // P5 (DIFFUSION3DPA_8): QDD0 = sum QQD0*Bt, QDD1 = sum QQD1*Gt, QDD2 = sum QQD2*Bt
  // over qy, column dx of plane qz.
  if (in2) {
    const int e = w / (Q * D), r = w % (Q * D), qz = r / D, dx = r % D;
    double* col = buf + e * K + qz * Q2 + dx;
    back(col, Q, 1, u);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int d = 0; d < D; ++d) col[k * Q3 + d * Q] = u[k][d];
  }
  __syncthreads();
  // P6 (DIFFUSION3DPA_9): sum over qz, Y += (u + v) + w.
  if (in1) {
    const int r = w % D2;
    back(buf + w / D2 * K + r / D * Q + r % D, Q2, 2, u);
#pragma unroll
    for (int dz = 0; dz < D; ++dz) yp[dz * D2] = y[dz] + ((u[0][dz] + u[1][dz]) + u[2][dz]);
  }
}

template <int D, int Q>
int launch_mass(const double* B, const double* Bt, const double* Dq, const double* X, double* Y, int64_t NE,
                hipStream_t s) {
  const int64_t grid = ceil_div(NE, MassShape<D, Q>::E);
  if (grid > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  mass3dpa_kernel<D, Q><<<dim3(unsigned(grid)), dim3(kBS), 0, s>>>(B, Bt, Dq, X, Y, NE);
  return launch_status();
}

template <int D, int Q>
int launch_mass_naive(const double* B, const double* Bt, const double* Dq, const double* X, double* Y, int64_t NE,
                      hipStream_t s) {
  if (NE > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  mass3dpa_naive_kernel<D, Q><<<dim3(unsigned(NE)), dim3(Q * Q), 0, s>>>(B, Bt, Dq, X, Y);
  return launch_status();
}

template <int D>
int mass_q(int q1d, bool naive, const double* B, const double* Bt, const double* Dq, const double* X, double* Y,
           int64_t NE, hipStream_t s) {
  if (q1d == D)
    return naive ? launch_mass_naive<D, D>(B, Bt, Dq, X, Y, NE, s) : launch_mass<D, D>(B, Bt, Dq, X, Y, NE, s);
  if (q1d == D + 1)
    return naive ? launch_mass_naive<D, D + 1>(B, Bt, Dq, X, Y, NE, s)
                 : launch_mass<D, D + 1>(B, Bt, Dq, X, Y, NE, s);
  if constexpr (D + 2 <= 9) {
    if (q1d == D + 2)
      return naive ? launch_mass_naive<D, D + 2>(B, Bt, Dq, X, Y, NE, s)
                   : launch_mass<D, D + 2>(B, Bt, Dq, X, Y, NE, s);
  }
  return RPX_ERR_UNSUPPORTED;
}

template <int D, bool SYMM>
int launch_diff(const double* B, const double* G, const double* Dq, const double* X, double* Y, int64_t NE,
                hipStream_t s) {
  constexpr int Q = D + 1;
  const int64_t grid = ceil_div(NE, kBS / (Q * Q));
  if (grid > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  diffusion3dpa_kernel<D, Q, SYMM><<<dim3(unsigned(grid)), dim3(kBS), 0, s>>>(B, G, Dq, X, Y, NE);
  return launch_status();
}

template <bool SYMM>
int diff_d(int d1d, const double* B, const double* G, const double* Dq, const double* X, double* Y, int64_t NE,
           hipStream_t s) {
  switch (d1d) {
    case 1: return launch_diff<1, SYMM>(B, G, Dq, X, Y, NE, s);
    case 2: return launch_diff<2, SYMM>(B, G, Dq, X, Y, NE, s);
    case 3: return launch_diff<3, SYMM>(B, G, Dq, X, Y, NE, s);
    case 4: return launch_diff<4, SYMM>(B, G, Dq, X, Y, NE, s);
    case 5: return launch_diff<5, SYMM>(B, G, Dq, X, Y, NE, s);
    case 6: return launch_diff<6, SYMM>(B, G, Dq, X, Y, NE, s);
    case 7: return launch_diff<7, SYMM>(B, G, Dq, X, Y, NE, s);
    case 8: return launch_diff<8, SYMM>(B, G, Dq, X, Y, NE, s);
    default: return RPX_ERR_UNSUPPORTED;
  }
}

}  // namespace

extern "C" {

int rpx_mass3dpa_f64(const double* B, const double* Bt, const double* D, const double* X, double* Y, int64_t NE,
                     int d1d, int q1d, const rpx_tuning* tune, void* stream) {
  if (NE < 0) return RPX_ERR_INVALID_ARGUMENT;
  if (NE == 0) return RPX_SUCCESS;
  if (!B || !Bt || !D || !X || !Y) return RPX_ERR_INVALID_ARGUMENT;
  hipStream_t s = as_stream(stream);
  const bool naive = (tune_flags(tune) & RPX_TUNE_NAIVE) != 0;
  switch (d1d) {
    case 1: return mass_q<1>(q1d, naive, B, Bt, D, X, Y, NE, s);
    case 2: return mass_q<2>(q1d, naive, B, Bt, D, X, Y, NE, s);
    case 3: return mass_q<3>(q1d, naive, B, Bt, D, X, Y, NE, s);
    case 4: return mass_q<4>(q1d, naive, B, Bt, D, X, Y, NE, s);
    case 5: return mass_q<5>(q1d, naive, B, Bt, D, X, Y, NE, s);
    case 6: return mass_q<6>(q1d, naive, B, Bt, D, X, Y, NE, s);
    case 7: return mass_q<7>(q1d, naive, B, Bt, D, X, Y, NE, s);
    case 8: return mass_q<8>(q1d, naive, B, Bt, D, X, Y, NE, s);
    default: return RPX_ERR_UNSUPPORTED;
  }
}

size_t rpx_mass3dpa_batched_scratch_bytes(const rpx_mass_batch* batches_host, int nbatch) {
  if (!batches_host || nbatch < 0) return 0;
  for (int i = 0; i < nbatch; ++i)
    if (batches_host[i].ne < 0 || batches_host[i].d1d < 1) return 0;
  return batch_layout(batches_host, nbatch).total;
}

int rpx_mass3dpa_batched_plan(const rpx_mass_batch* batches_host, int nbatch, void* scratch, size_t scratch_bytes,
                              void* stream) {
  if (!batches_host || nbatch < 0 || !scratch) return RPX_ERR_INVALID_ARGUMENT;
  for (int i = 0; i < nbatch; ++i) {
    const rpx_mass_batch& b = batches_host[i];
    if (b.ne < 0 || (b.ne > 0 && (!b.B || !b.Bt || !b.D || !b.X || !b.Y))) return RPX_ERR_INVALID_ARGUMENT;
    if (b.d1d < 1 || b.d1d > 8 || b.q1d != b.d1d + 1) return RPX_ERR_UNSUPPORTED;
  }
  const BatchLayout l = batch_layout(batches_host, nbatch);
  if (scratch_bytes < l.total) return RPX_ERR_SCRATCH_TOO_SMALL;
  if (l.nchunks > INT32_MAX) return RPX_ERR_UNSUPPORTED;
  forget_plan(scratch);  // recorded again once the new tables are uploaded
  // Chunks of the highest orders (the costliest) come first, so that the
  // persistent workgroups end on cheap chunks; a batch's chunks stay
  // contiguous.
  std::vector<int> order(static_cast<size_t>(nbatch));
  for (int i = 0; i < nbatch; ++i) order[size_t(i)] = i;
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int b) { return batches_host[a].d1d > batches_host[b].d1d; });
  std::vector<int> chunk_batch(size_t(l.nchunks));
  std::vector<int64_t> chunk0(size_t(nbatch + 1));
  int64_t c = 0;
  for (int i : order) {
    chunk0[size_t(i)] = c;
    const int64_t k = ceil_div(batches_host[i].ne, batch_chunk_elems(batches_host[i].d1d));
    for (int64_t j = 0; j < k; ++j) chunk_batch[size_t(c + j)] = i;
    c += k;
  }
  chunk0[size_t(nbatch)] = c;
  BatchHeader h{};
  h.nchunks = l.nchunks;
  h.nbatch = nbatch;
  for (int i : order) {
    const int d = batches_host[i].d1d;
    const int64_t first = chunk0[size_t(i)];
    const int64_t last = first + ceil_div(batches_host[i].ne, batch_chunk_elems(d));
    if (h.order_end[d] == h.order_begin[d]) h.order_begin[d] = first;  // first batch of this order
    h.order_end[d] = last;
  }
  hipStream_t st = as_stream(stream);
  char* base = reinterpret_cast<char*>(scratch);
  RPX_TRY(hipMemcpyAsync(base, &h, sizeof(h), hipMemcpyHostToDevice, st));
  if (nbatch > 0)
    RPX_TRY(hipMemcpyAsync(base + l.batches_off, batches_host, size_t(nbatch) * sizeof(rpx_mass_batch),
                           hipMemcpyHostToDevice, st));
  if (l.nchunks > 0)
    RPX_TRY(hipMemcpyAsync(base + l.chunk_batch_off, chunk_batch.data(), chunk_batch.size() * sizeof(int),
                           hipMemcpyHostToDevice, st));
  RPX_TRY(hipMemcpyAsync(base + l.chunk0_off, chunk0.data(), chunk0.size() * sizeof(int64_t),
                         hipMemcpyHostToDevice, st));
  RPX_TRY(hipStreamSynchronize(st));  // the host tables must outlive the copies
  int64_t chunks[9];
  for (int d = 0; d < 9; ++d) chunks[d] = h.order_end[d] - h.order_begin[d];
  record_plan(scratch, chunks);
  return RPX_SUCCESS;
}

int rpx_mass3dpa_batched_run(const void* scratch, const rpx_tuning* tune, void* stream) {
  if (!scratch) return RPX_ERR_INVALID_ARGUMENT;
  int dev = 0, cus = 0;
  RPX_TRY(hipGetDevice(&dev));
  RPX_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const char* plan = reinterpret_cast<const char*>(scratch);
  hipStream_t s = as_stream(stream);
  const int64_t grid_override = tune_or(tune, &rpx_tuning::grid_size, 0);
  if ((tune_flags(tune) & RPX_TUNE_MASS_SINGLE_LAUNCH) == 0) {
    int rc = RPX_SUCCESS;
    int64_t chunks[9];
    if (grid_override == 0 && find_plan(scratch, chunks)) {
      // One launch per order present, one workgroup per chunk, highest first.
      if (rc == RPX_SUCCESS) rc = launch_order_chunks<8>(plan, chunks[8], s);
      if (rc == RPX_SUCCESS) rc = launch_order_chunks<7>(plan, chunks[7], s);
      if (rc == RPX_SUCCESS) rc = launch_order_chunks<6>(plan, chunks[6], s);
      if (rc == RPX_SUCCESS) rc = launch_order_chunks<5>(plan, chunks[5], s);
      if (rc == RPX_SUCCESS) rc = launch_order_chunks<4>(plan, chunks[4], s);
      if (rc == RPX_SUCCESS) rc = launch_order_chunks<3>(plan, chunks[3], s);
      if (rc == RPX_SUCCESS) rc = launch_order_chunks<2>(plan, chunks[2], s);
      if (rc == RPX_SUCCESS) rc = launch_order_chunks<1>(plan, chunks[1], s);
      if (rc != RPX_SUCCESS) return rc;
      // The chunks beyond those grids: none when the record matches the
      // plan in scratch; the rest of a larger plan written there since by
      // other means (a copy into a reused address).
      ChunkSkip skip;
      std::copy(chunks, chunks + 9, skip.done);
      mass3dpa_batched_kernel<<<dim3(unsigned(cus)), dim3(kBS), 0, s>>>(plan, skip);
      return launch_status();
    }
    // One persistent launch per order, highest first (the plan's order).
    if (rc == RPX_SUCCESS) rc = launch_order<8>(plan, cus, grid_override, s);
    if (rc == RPX_SUCCESS) rc = launch_order<7>(plan, cus, grid_override, s);
    if (rc == RPX_SUCCESS) rc = launch_order<6>(plan, cus, grid_override, s);
    if (rc == RPX_SUCCESS) rc = launch_order<5>(plan, cus, grid_override, s);
    if (rc == RPX_SUCCESS) rc = launch_order<4>(plan, cus, grid_override, s);
    if (rc == RPX_SUCCESS) rc = launch_order<3>(plan, cus, grid_override, s);
    if (rc == RPX_SUCCESS) rc = launch_order<2>(plan, cus, grid_override, s);
    if (rc == RPX_SUCCESS) rc = launch_order<1>(plan, cus, grid_override, s);
    return rc;
  }
  // One persistent launch for all orders: workgroups per CU times CUs
  // (tune->grid_size overrides); workgroups beyond the chunk count exit at
  // once.  The kernel finds the tables from the counts in the plan's header.
  const int64_t grid = grid_override > 0 ? grid_override : 3 * int64_t(cus);
  if (grid > INT32_MAX) return RPX_ERR_INVALID_ARGUMENT;
  mass3dpa_batched_kernel<<<dim3(unsigned(grid)), dim3(kBS), 0, s>>>(plan, ChunkSkip{});
  return launch_status();
}

int rpx_mass3dpa_batched_f64(const rpx_mass_batch* batches_host, int nbatch, void* scratch, size_t scratch_bytes,
                             const rpx_tuning* tune, void* stream) {
  const int rc = rpx_mass3dpa_batched_plan(batches_host, nbatch, scratch, scratch_bytes, stream);
  if (rc != RPX_SUCCESS) return rc;
  return rpx_mass3dpa_batched_run(scratch, tune, stream);
}

int rpx_diffusion3dpa_f64(const double* Basis, const double* dBasis, const double* D, const double* X, double* Y,
                          int64_t NE, int d1d, int q1d, int symmetric, const rpx_tuning* /*tune*/, void* stream) {
  if (NE < 0) return RPX_ERR_INVALID_ARGUMENT;
  if (NE == 0) return RPX_SUCCESS;
  if (!Basis || !dBasis || !D || !X || !Y) return RPX_ERR_INVALID_ARGUMENT;
  if (q1d != d1d + 1) return RPX_ERR_UNSUPPORTED;
  hipStream_t s = as_stream(stream);
  return symmetric ? diff_d<true>(d1d, Basis, dBasis, D, X, Y, NE, s)
                   : diff_d<false>(d1d, Basis, dBasis, D, X, Y, NE, s);
}

}  // extern "C"
