// Mixed-precision sparse GAP kernel on the gfx950 matrix cores: BF16 hi+lo
// split operands (x = hi + lo, three products hi.hi + hi.lo + lo.hi) with
// FP32 accumulation, fused zeta-power / energy / weight epilogue.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "device_buffer.hh"
#include "gap_kernels.hh"

namespace rgpu {

// Sparse points in the packed layout of the invariants (packing.hh),
// pre-split into BF16 hi/lo planes, in the two layouts the two GEMMs read:
// [M][D] (K-contiguous rows for K = X T^T) and [D][Mp] (K-contiguous
// columns for T~ = W~ T, the points of species s in columns col[s] on, each
// species padded with zero columns to a multiple of 32); D here is the
// packed width.
struct MixedSparse {
  int64_t D = 0, Mp = 0;
  std::vector<int64_t> col;
  DeviceBuffer<unsigned short> t_hi, t_lo;    // [M][D]
  DeviceBuffer<unsigned short> tt_hi, tt_lo;  // [D][Mp]
};

// A BF16 hi/lo pair of planes (same shape); bit patterns of __bf16.
struct SplitPlanes {
  unsigned short* hi = nullptr;
  unsigned short* lo = nullptr;
};

bool mfma_available();
// T: [M][D] FP64 rows (device) in the full layout of S species, N radial
// channels, L1 = max_angular + 1; rows [sp_off[s], sp_off[s + 1]) belong to
// species s
void prepare_mixed_sparse(MixedSparse& ms, const double* T, int64_t M, int S, int N, int L1,
                          const std::vector<int64_t>& sp_off, hipStream_t stream);
// row stride of the W~ planes of a block of n_cols sparse points: n_cols
// rounded up to the K step of the force product, pad columns zero
int64_t gap_mixed_wt_stride(int64_t n_cols);
// K tile GEMM + epilogue for all species blocks in grouped launches.  The
// features are given split: X = xs.hi + xs.lo, [n_centres][D] (rows gathered
// through the blocks' row_idx, un-normalised, scaled by 1/|p| in the
// epilogue).  Outputs: energy (of the blocks with sparse points, per centre;
// summed over the column tiles through part, [gap_mixed_energy_tiles of the
// blocks' row and column counts] x [ld >= n_centres] doubles, see EnergyTiles)
// and the weighted kernel gradient W~ of each block, split,
// [n_rows][gap_mixed_wt_stride(n_cols)] (wts may be null).
int gap_mixed_energy_tiles(const int64_t* rows, const int64_t* cols, int n_blocks, int64_t ld);
void run_gap_mixed_kernel(const GapBlock<float>* blks, int n_blocks, const MixedSparse& ms,
                          SplitPlanes xs, double* energy, double* part, int64_t ld, const SplitPlanes* wts,
                          hipStream_t stream);
// T~ rows: G[row_idx[r]][:] = sum_m W~_b[r][m] T[col0+m][:]; block b holds
// the sparse points of species b
void run_gap_mixed_force(const GapBlock<float>* blks, int n_blocks, const MixedSparse& ms,
                         const SplitPlanes* wts, float* G, hipStream_t stream);

}  // namespace rgpu
