// FP64 GAP GEMMs on the gfx950 matrix cores (parity path).
#pragma once

#include <hip/hip_runtime.h>

#include "gap_kernels.hh"

namespace rgpu {

// contraction lengths are padded to the K step: feature rows (the blocks' D)
// and W~ rows hold zeros from their last column up to this stride
int64_t gap_f64_k_stride(int64_t k);

// K GEMM + epilogue for all species blocks (grouped): energy per centre (of
// the blocks with sparse points; summed over the column tiles through part,
// [gap_f64_energy_tiles(n_cols) of the widest block] x [ld >= n_centres]
// doubles, see EnergyTiles) and
// wts[b] [n_rows][gap_f64_k_stride(n_cols)] (wts may be null)
int gap_f64_energy_tiles(int64_t n_cols);
void run_gap_f64_kernel(const GapBlock<double>* blks, int n_blocks, double* energy, double* part, int64_t ld,
                        double* const* wts, hipStream_t stream);
// out[row_idx[r] * ld + col0 + m] = (X_r . T_m)^zeta of every block
void run_gap_f64_rows(const GapBlock<double>* blks, int n_blocks, double* out, int64_t ld, hipStream_t stream);
// dL/dp rows G[row_idx[r]][:] from dL/dX_r = sum_m wts[b][r][m] T[col0+m][:]:
// dL/dX itself for features that are not normalised, else with the
// normalisation's transpose, dL/dX / |p| - (X . dL/dX) p / |p|^2, X . dL/dX =
// xg_scale xg[centre] (in the product's epilogue, where the row of p is one
// read beside a compute-bound kernel)
void run_gap_f64_force(const GapBlock<double>* blks, int n_blocks, double* const* wts, const double* xg,
                       double xg_scale, double* G, hipStream_t stream);

// C (n x n) = A^T A for A [rows][n] (device pointers; Ap: room for rows x (n +
// 1) doubles when n is odd, else not used; At: room for n x
// gap_f64_k_stride(rows) doubles; iota: 0 .. n-1 as ints)
void run_gram_f64(int64_t rows, int64_t n, const double* A, double* Ap, double* At, const int* iota, double* C,
                  hipStream_t stream);

}  // namespace rgpu
