// Power spectrum in symmetric packed rows, and its adjoint to dL/dc.
//
// The expansion of a centre is, per angular channel l, a matrix C_l of
// R = S N rows (species-major, then radial channel) and 2l+1 columns, and its
// power spectrum is the symmetric matrix f_l C_l C_l^T, f_l = (2l+1)^{-1/2}.
// A symmetric packed row holds, l by l, the upper triangle of that matrix by
// columns: entry (r, c), r <= c, at l TRI + c (c + 1) / 2 + r with
// TRI = R (R + 1) / 2, the entries r < c times sqrt 2, and zero columns up to
// a multiple of 32.  A dot product of two such rows equals the dot product of
// the full feature rows (keys a <= b, [n1][n2][l]) when one of them is a
// feature row; for another vector t the entries of a diagonal key are
// (t[n1][n2] + t[n2][n1]) / sqrt 2 (n1 < n2) and t[n][n]; of two such vectors
// it is the product of their symmetric parts only.  A row is as short as
// the key-major packed row (packing.hh), but an angular channel is one
// contiguous run, so a wavefront can take a channel with a lane per row r and
// every other operand wavefront-uniform.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_buffer.hh"

namespace rgpu {

__host__ __device__ inline int64_t sym_tri(int64_t r) { return r * (r + 1) / 2; }
__host__ __device__ inline int64_t sym_row_stride(int S, int N, int L1) {
  return (int64_t(L1) * sym_tri(int64_t(S) * N) + 31) / 32 * 32;
}

// p[i] = the symmetric packed row of c[i] (c [n][S][N][(L+1)^2]),
// un-normalised, pad columns zero; norm2[i] = |p[i]|^2
void launch_sym_power(int S, int N, int L1, int64_t n, const double* c, double* p, double* norm2,
                      hipStream_t stream);

// dL/dc of each centre, written [n][S][(L+1)^2][N], from dL/dp in symmetric
// packed rows
void launch_sym_contract(int S, int N, int L1, int64_t n, const double* c, const double* G, double* dc,
                         hipStream_t stream);
// the same from dL/dX, X = p / |p|, in symmetric packed rows: p likewise, xg[i] =
// X . dL/dX
void launch_sym_contract_projected(int S, int N, int L1, int64_t n, const double* c, const double* p,
                                   const double* norm2, const double* xg, const double* G, double* dc,
                                   hipStream_t stream);
// dL/dc [n_sets][n_ids] of the kernel derivatives of sparse points T (symmetric
// packed rows, one per set) at the centres ids: dL/dX_i = zeta d^(zeta - 1) T_q
// with d = X_i . T_q = dot[i ld_dot + q], X = p / |p|; E: dL/dc of dL/dp = p for
// every centre of the batch (launch_sym_contract; null: X = p)
struct SymSets {
  const int* ids = nullptr;
  int64_t n_ids = 1;
  const double* dot = nullptr;
  int64_t ld_dot = 0;
  int zeta = 1;
};
void launch_sym_contract_sets(int S, int N, int L1, int64_t n_sets, const SymSets& sets, const double* c,
                              const double* norm2, const double* E, const double* T, double* dc, hipStream_t stream);
// dL/dc of each centre, as launch_sym_contract, from dL/dX in full rows
// [n][K N^2 (L+1)] (keys a <= b): X = p / |p| with p in symmetric packed rows,
// or X = p (p null).  work: packed rows where they are needed
void launch_sym_contract_full(int S, int N, int L1, int64_t n, const double* c, const double* p, const double* norm2,
                              const double* G, DeviceBuffer<double>& work, double* dc, hipStream_t stream);

// Full rows [.][K N^2 (L+1)] to symmetric packed rows and back.  Packing row
// r from full row rows[r] (rows null: row r); unpacking row r of out from
// packed row rows[r], divided by its norm when normalising.  asymmetric (may
// be null): set to 1 when a diagonal key's block of a full row is not symmetric
// (such a row is not recovered from its packed one).
void launch_sym_pack(int S, int N, int L1, int64_t n, const double* full, const int64_t* rows, double* out,
                     hipStream_t stream, int* asymmetric = nullptr);
void launch_sym_unpack(int S, int N, int L1, int64_t n, const double* p, const int64_t* rows, const double* norm2,
                       bool normalize, double* out, hipStream_t stream);

}  // namespace rgpu
