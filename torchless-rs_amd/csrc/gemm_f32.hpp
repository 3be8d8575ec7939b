// The order in which every product of the plain path adds (gemm_plain.hip), and the tiles of 32-bit operands (gemm_f32.hip).
#pragma once
#include "common.hpp"

namespace tl {

constexpr int PG = 8, PR = 8;                     // groups of K, runs of a group
constexpr int BK = 16;                            // runs are a multiple of this long

// A launch has fewer than 2^32 threads along x (more are not refused: some are left out), here 512 a workgroup; what has more
// workgroups goes on along another dimension.
constexpr long GRID_X = 1l << 22;

__host__ __device__ __forceinline__ int run_length(int K) { return (K + PG * PR * BK - 1) / (PG * PR * BK) * BK; }

// Can the tiles on the matrix cores take these operands?
bool f32_tiles_fit(const float* A, const float* W, int K, int lda, int ldw);
// Over how many workgroups a tile's groups of K are dealt; more than 1: `parts` [PG][M][N] receives the groups' sums on their way.
int f32_tiles_split(int M, int N, int K);
int f32_tiles(const float* A, const float* W, float* C, float* parts, int M, int N, int K, int lda, int ldw, int ldc, int accumulate, hipStream_t st);

}  // namespace tl
