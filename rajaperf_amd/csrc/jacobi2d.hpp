// JACOBI_2D on register-resident tiles (jacobi2d_block.hip).
#pragma once

#include "rpx_common.hpp"

namespace rpx {

// Largest grid that one workgroup holds.
constexpr int64_t kJacobiOneTileN = 128;

// `tsteps` >= 1 time steps of a grid of 3 <= N <= kJacobiOneTileN, in one launch.
int jacobi_one_tile(double* A, double* B, int64_t N, int64_t tsteps, hipStream_t s);

// `tsteps` >= 2 time steps of a grid of N > kJacobiOneTileN, even or odd, with
// the N x N grid Q as scratch; 8-byte alignment.  RPX_ERR_UNSUPPORTED, before
// anything is launched, where no tile shape fits.
int jacobi_blocks(double* A, double* B, double* Q, int64_t N, int64_t tsteps, hipStream_t s);

}  // namespace rpx
