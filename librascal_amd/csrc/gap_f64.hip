// FP64 GAP GEMMs on the gfx950 matrix cores (v_mfma_f64_16x16x4_f64), the
// parity path of the sparse GAP prediction.
//
//   kernel:  K[r][m] = sum_d X[row(r)][d] T[col0+m][d]   (B rows K-contiguous)
//   rows:    the same, K^zeta stored as K_NM rows
//   forces:  G[row(r)][d] = sum_m W~[r][m] T[col0+m][d]  (B given as [K][N])
//
// Tiling: 256 threads, block tiles of 64 x 64 (wavefronts 2 x 2, 32 x 32
// each), 32 x 64 (16 x 32 each) or 16 x 64 (wavefronts 1 x 4) by the number
// of tiles (launch below), K step 16.  Rows are 16-byte aligned and K a multiple of 16 (zero
// pads), so every operand goes straight to LDS (global_load_lds_dwordx4) in
// NS = 3 stages with two K steps in flight and one barrier per step.  A step
// is short (0.1 - 0.2 us of products), so what bounds the kernel away from the
// matrix cores is the latency of its loads: the waits are counted by hand and
// the barrier is the bare instruction (__syncthreads would drain every load
// in flight), and the stages are passed to the tile function by reference (on
// arrays of the kernel itself the compiler waits for all loads before each
// LDS read).  8192-long products of the GAP shapes, 4096 x 512 x 11776: 62.9
// TFLOP/s (64 x 64 tiles 56.9; with drained barriers 47.1; the register-staged
// kernel before 45); 1024 x 512 x 11776: 45.9 (64 x 64: 27.7, drained 17.9);
// 512 x 512 x 11776: 23.6 and 32.4 in half-size tiles.
//
// A K step of a K-contiguous operand is 64 rows x 128 B; row r of a group of
// 8 keeps its 16-byte chunk q at slot 8 r + (q ^ r), so 8 rows' reads of one
// chunk hit distinct banks.  A chunk holds two K values: lane group
// fq = lane / 16 reads chunk 4 h + fq for the products (h, e), e = 0, 1, so
// product (h, e) contracts K values 2 (4 h + fq) + e; the force product's B
// rows (k, 64 columns, read 8 bytes at a time along the row) follow the same
// numbering.
//
// Grouped launch over species blocks, tiles dealt to the XCDs as the mixed-
// precision kernel's (groups of kGroupM row panels walked column by column, a
// contiguous range of them per XCD, so the tiles resident on one XCD share
// operand panels through its L2).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hh"
#include "gap_f64.hh"

namespace rgpu {

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(double)))) double f64x4;
typedef __attribute__((__vector_size__(2 * sizeof(double)))) double f64x2;

constexpr int BN = 64, BK = 16, NT = 256, NS = 3;
constexpr int kMaxProblems = 16;
constexpr int kGroupM = 8;  // row panels per tile group

struct Problem {
  int64_t M, N, K;   // K a multiple of BK
  int64_t Kv;        // force form: rows of B (K rows past them read zeros, as A's pads)
  const double* A;
  int64_t lda;
  const int* a_rows;
  const double* B;   // kernel: rows n (K contiguous); force: rows k (N contiguous)
  int64_t ldb;
  const int* c_rows;
  int64_t tile0;
  int tiles_m, tiles_n;
  const double* norm2;
  const double* alpha;
  double* epart;  // energy partials [tiles_n][ldp], by centre
  int64_t ldp;
  double* wt;     // [M][ldw], columns N .. ldw zero
  int64_t ldw;
  double* G;
  int64_t ldg;
  const double* xp;  // force form: X rows [centre][ldg] projected out of G (may be null)
  const double* xg;  // [centre] X . dL/dX / scale
};

struct ProblemSet {
  Problem p[kMaxProblems];
  int64_t total_tiles;
  int n;
  int normalize;
  int zeta;
  double xg_scale;
};

__device__ __forceinline__ double pow_int(double v, int n) {
  if (n == 0) return 1.0;
  if (n == 1) return v;
  if (n == 2) return v * v;
  if (n == 3) return v * v * v;
  double r = 1.0, x = v;
  unsigned u = unsigned(n);
  do {
    if (u & 1) r *= x;
    u >>= 1;
    x *= x;
  } while (u);
  return r;
}

// s_waitcnt vmcnt(N) lgkmcnt(0) (gfx9 encoding)
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}
__device__ __forceinline__ void bare_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// the K rows past the last sparse point of a force product
__device__ double zero_row[BN];

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 raw16;  // 16 bytes

template <int BM>
struct Stages {
  raw16 A[NS][BM * BK / 2];
  raw16 B[NS][BN * BK / 2];
  double esum[4][BM];  // row sums of the wavefronts along N
};

// EPI 0: W~ and energy partials; 1: force rows of G; 2: K^zeta rows into G.
// WM x WN wavefronts of 16 TI x 16 TJ outputs each.
template <int EPI, int WM, int TI, int TJ>
__device__ __forceinline__ void gemm_tile(const ProblemSet& ps, const Problem& P, int64_t tm, int64_t tn,
                                          Stages<16 * WM * TI>& sm) {
  constexpr int BM = 16 * WM * TI, WN = 4 / WM;
  static_assert(WN * 16 * TJ == BN, "the wavefronts cover the tile's columns");
  const int64_t r0 = tm * BM, c0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave - wm * WN;

  // Loads of one K step, 64 lanes x 16 B each: A rows in BM / 8 instructions
  // (dealt to the wavefronts), B in eight (two per wavefront).
  // K-contiguous: lane l takes row l / 8 of a group of 8 and the chunk its
  // slot holds; B of the force form: row k = l / 32 of a pair of K rows,
  // chunk l % 32.  Rows and columns past the matrix repeat its last ones
  // (their results are never stored).
  constexpr int GA = BM / 8, LA = (GA + 3) / 4;
  auto a_group = [&](int j) { return GA >= 4 ? wave + 4 * j : (wave < GA ? wave : 0); };
  const int rr = lane >> 3, qq = (lane & 7) ^ rr;
  const int64_t nk = P.K / BK;
  const double *pa[LA], *pb[2];
  bool pad[2] = {false, false};  // force form: this lane's row of the last K step is a pad
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    int64_t ra = r0 + a_group(j) * 8 + rr;
    ra = ra < P.M ? ra : P.M - 1;
    if (P.a_rows) ra = P.a_rows[ra];
    pa[j] = P.A + ra * P.lda + 2 * qq;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (EPI != 1) {
      int64_t rb = c0 + (wave + 4 * j) * 8 + rr;
      rb = rb < P.N ? rb : P.N - 1;
      pb[j] = P.B + rb * P.ldb + 2 * qq;
    } else {
      int64_t cb = c0 + 2 * (lane & 31);
      cb = cb + 2 <= P.ldb ? cb : P.ldb - 2;
      const int64_t kb = (wave + 4 * j) * 2 + (lane >> 5);  // row of a K step
      pb[j] = P.B + kb * P.ldb + cb;
      pad[j] = kb + (nk - 1) * BK >= P.Kv;
    }
  }
  auto issue = [&](int s, int64_t kt) {
    const int64_t ks = kt < nk ? kt : nk - 1, k = ks * BK;  // surplus loads land in stages never read
    // (every wavefront counts the same loads: with fewer row groups than
    // wavefronts, the others store the first group's values once more)
#pragma unroll
    for (int j = 0; j < LA; ++j)
      __builtin_amdgcn_global_load_lds(pa[j] + k, &sm.A[s][a_group(j) * 64], 16, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int g = (wave + 4 * j) * 64;
      if (EPI != 1) {
        __builtin_amdgcn_global_load_lds(pb[j] + k, &sm.B[s][g], 16, 0, 0);
      } else {
        const double* src = ks == nk - 1 && pad[j] ? zero_row + 2 * (lane & 31) : pb[j] + k * P.ldb;
        __builtin_amdgcn_global_load_lds(src, &sm.B[s][g], 16, 0, 0);
      }
    }
  };

  f64x4 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0;

  const int fr = lane & 15, fq = lane >> 4;
  // slot of chunk q of row r
  auto slot = [&](int r, int q) { return (r >> 3) * 64 + (r & 7) * 8 + (q ^ (r & 7)); };
  auto compute = [&](int s) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f64x2 a[TI], b[TJ];
#pragma unroll
      for (int i = 0; i < TI; ++i)
        a[i] = __builtin_bit_cast(f64x2, sm.A[s][slot((wm * TI + i) * 16 + fr, 4 * h + fq)]);
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int n = (wn * TJ + j) * 16 + fr;
        if (EPI != 1) {
          b[j] = __builtin_bit_cast(f64x2, sm.B[s][slot(n, 4 * h + fq)]);
        } else {
          const double* row = reinterpret_cast<const double*>(sm.B[s]) + 2 * (4 * h + fq) * BN + n;
          b[j][0] = row[0];
          b[j][1] = row[BN];
        }
      }
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
    }
  };

  constexpr int PER = LA + 2;  // load instructions per wavefront and K step
  if (nk > 0)
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) issue(s, s);
  int s_read = 0, s_fill = NS - 1;
  for (int64_t kt = 0; kt < nk; ++kt) {
    // this wavefront's loads of step kt are done once at most the later
    // steps' remain; the barrier extends that to every wavefront and orders
    // the previous step's reads (done: lgkmcnt 0) before the refill of its
    // stage
    wait_loads<(NS - 2) * PER>();
    bare_barrier();
    issue(s_fill, kt + NS - 1);
    compute(s_read);
    s_read = s_read + 1 == NS ? 0 : s_read + 1;
    s_fill = s_fill + 1 == NS ? 0 : s_fill + 1;
  }
  wait_loads<0>();  // no load may still write this workgroup's LDS when it exits

  // element e of a 16x16 tile: row lane/16 + 4*e, column lane%16
  if (EPI == 0 || EPI == 2) {
    double rowsum[TI][4];
#pragma unroll
    for (int ie = 0; ie < 4 * TI; ++ie) {
      const int i = ie >> 2, e = ie & 3;
      rowsum[i][e] = 0.0;
      const int64_t r = r0 + (wm * TI + i) * 16 + fq + 4 * e;
      if (r >= P.M) continue;
      const int centre = P.c_rows[r];
      double inv = 1.0;
      if (ps.normalize) {
        const double n2 = P.norm2[centre];
        inv = n2 > 0 ? 1.0 / sqrt(n2) : 1.0;
      }
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int64_t c = c0 + (wn * TJ + j) * 16 + fr;
        const double k = acc[i][j][e] * inv;
        if (EPI == 2) {
          if (c < P.N) P.G[int64_t(centre) * P.ldg + c] = pow_int(k, ps.zeta);
          continue;
        }
        if (c >= P.N) {
          if (P.wt && c < P.ldw) P.wt[r * P.ldw + c] = 0.0;
          continue;
        }
        const double a = P.alpha[c];
        rowsum[i][e] += a * pow_int(k, ps.zeta);
        if (P.wt) P.wt[r * P.ldw + c] = a * (ps.zeta > 1 ? ps.zeta * pow_int(k, ps.zeta - 1) : 1.0);
      }
    }
    if (EPI == 2) return;
#pragma unroll
    for (int ie = 0; ie < 4 * TI; ++ie) {
      const int i = ie >> 2, e = ie & 3;
      double v = rowsum[i][e];
      for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
      if (fr == 0) sm.esum[wn][(wm * TI + i) * 16 + fq + 4 * e] = v;
    }
    __syncthreads();
    if (P.epart && tid < BM) {
      const int64_t r = r0 + tid;
      double t = 0.0;
#pragma unroll
      for (int w = 0; w < WN; ++w) t += sm.esum[w][tid];
      if (r < P.M) P.epart[tn * P.ldp + P.c_rows[r]] = t;
    }
  } else {
#pragma unroll
    for (int ie = 0; ie < 4 * TI; ++ie) {
      const int i = ie >> 2, e = ie & 3;
      const int64_t r = r0 + (wm * TI + i) * 16 + fq + 4 * e;
      if (r >= P.M) continue;
      const int centre = P.c_rows[r];
      double* g = P.G + int64_t(centre) * P.ldg;
      double alpha = 1.0, beta = 0.0;
      if (P.xp) {
        const double n2 = P.norm2[centre];
        if (n2 > 0) {
          alpha = 1.0 / sqrt(n2);
          beta = ps.xg_scale * P.xg[centre] / n2;
        }
      }
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int64_t c = c0 + (wn * TJ + j) * 16 + fr;
        if (c >= P.N) continue;
        double v = acc[i][j][e];
        if (P.xp) v = alpha * v - beta * P.xp[int64_t(centre) * P.ldg + c];
        g[c] = v;
      }
    }
  }
}

template <int EPI, int WM, int TI, int TJ>
__global__ __launch_bounds__(NT, TI == 2 ? 3 : 4) void f64_gemm(ProblemSet ps) {
  // the workgroups go to the 8 XCDs round robin: XCD x takes linear tiles
  // [x per_xcd, (x + 1) per_xcd)
  const int64_t per_xcd = (int64_t(gridDim.x) + 7) / 8;
  const int64_t bid = int64_t(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (bid >= ps.total_tiles) return;  // whole workgroup, before any barrier
  int pi = 0;
  while (pi + 1 < ps.n && bid >= ps.p[pi + 1].tile0) ++pi;
  const Problem& P = ps.p[pi];
  const int64_t local = bid - P.tile0;
  const int64_t per_group = int64_t(kGroupM) * P.tiles_n;
  const int64_t grp = local / per_group, in = local - grp * per_group;
  const int64_t gm = std::min<int64_t>(kGroupM, P.tiles_m - grp * kGroupM);
  const int64_t tn = in / gm;
  __shared__ __align__(16) Stages<16 * WM * TI> sm;
  gemm_tile<EPI, WM, TI, TJ>(ps, P, grp * kGroupM + (in - tn * gm), tn, sm);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int64_t layout_tiles(ProblemSet& ps, int bm) {
  int64_t tiles = 0;
  for (int i = 0; i < ps.n; ++i) {
    Problem& P = ps.p[i];
    P.tile0 = tiles;
    P.tiles_m = int((P.M + bm - 1) / bm);
    P.tiles_n = int((P.N + BN - 1) / BN);
    tiles += int64_t(P.tiles_m) * P.tiles_n;
  }
  return tiles;
}

template <int EPI>
void launch(ProblemSet& ps, hipStream_t stream) {
  for (int i = 0; i < ps.n; ++i) {
    const Problem& P = ps.p[i];
    if (P.K % BK != 0 || P.lda % 2 != 0 || P.ldb % 2 != 0 || !aligned16(P.A) || !aligned16(P.B))
      throw InvalidArgument("internal: unaligned operands of the FP64 GAP product");
  }
  // 64-row tiles from 2048 tiles (eight per CU) up, where the operand traffic
  // of smaller ones through L2 costs more than their better balance gives
  // (4096 x 11776 x 512 forces: 1.02 ms in 32-row tiles, 9 GB); 32-row tiles
  // down to one per CU (4096 x 512 x 11776: 0.79 ms against 0.87 in 64-row
  // tiles; 1024 x 512 x 11776: 0.269 ms against 0.282 in 16-row tiles), then
  // 16-row ones (512 x 512 x 11776: 0.19 ms against 0.26).
  int rows = 64;
  if (layout_tiles(ps, 64) < 2048) rows = layout_tiles(ps, 32) < 256 ? 16 : 32;
  ps.total_tiles = layout_tiles(ps, rows);
  if (ps.total_tiles == 0) return;
  const unsigned grid = unsigned((ps.total_tiles + 7) / 8 * 8);  // whole rounds over the 8 XCDs
  if (rows == 64)
    hipLaunchKernelGGL((f64_gemm<EPI, 2, 2, 2>), dim3(grid), dim3(NT), 0, stream, ps);
  else if (rows == 32)
    hipLaunchKernelGGL((f64_gemm<EPI, 2, 1, 2>), dim3(grid), dim3(NT), 0, stream, ps);
  else
    hipLaunchKernelGGL((f64_gemm<EPI, 1, 1, 1>), dim3(grid), dim3(NT), 0, stream, ps);
  RGPU_LAUNCH_CHECK();
}

// out[c * ldo + r] = in[r * cols + c] for r < rows, c < cols, 32 x 32 tiles
// through LDS; padded (may be null): the rows of in again, cols + 1 apart with a
// zero at their end.  (Rows of an odd length are moved apart here: copied apart
// from the host row by row, a 1001 x 333 matrix took 9.5 ms, and apart on the
// device by a copy of its own 0.41 ms, against 0.30 ms this way.)
__global__ void transpose_f64_kernel(int64_t rows, int64_t cols, const double* __restrict__ in,
                                     double* __restrict__ out, int64_t ldo, double* __restrict__ padded) {
  __shared__ double t[32][33];
  const int64_t r0 = int64_t(blockIdx.y) * 32, c0 = int64_t(blockIdx.x) * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8 threads
  for (int k = ty; k < 32; k += 8) {
    const int64_t r = r0 + k, c = c0 + tx;
    if (r < rows && c < cols) {
      const double v = in[r * cols + c];
      t[k][tx] = v;
      if (padded) {
        padded[r * (cols + 1) + c] = v;
        if (c == cols - 1) padded[r * (cols + 1) + cols] = 0.0;
      }
    }
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int64_t c = c0 + k, r = r0 + tx;
    if (r < rows && c < cols) out[c * ldo + r] = t[tx][k];
  }
}

}  // namespace

int64_t gap_f64_k_stride(int64_t k) { return (k + BK - 1) / BK * BK; }

int gap_f64_energy_tiles(int64_t n_cols) { return int((n_cols + BN - 1) / BN); }

namespace {

// the kernel form of block b: rows X, columns T of the block
void kernel_problem(Problem& P, const GapBlock<double>& blk) {
  P.M = blk.n_rows;
  P.N = blk.n_cols;
  P.K = P.Kv = blk.D;
  P.A = blk.X;
  P.lda = blk.D;
  P.a_rows = blk.row_idx;
  P.B = blk.Tm + blk.col0 * blk.D;
  P.ldb = blk.D;
  P.c_rows = blk.row_idx;
  P.norm2 = blk.norm2;
}

}  // namespace

void run_gap_f64_kernel(const GapBlock<double>* blks, int n_blocks, double* energy, double* part, int64_t ld,
                        double* const* wts, hipStream_t stream) {
  static_assert(kMaxProblems <= EnergyTiles::kMax, "one energy reduction per grouped launch");
  for (int b0 = 0; b0 < n_blocks; b0 += kMaxProblems) {
    ProblemSet ps{};
    EnergyTiles et;
    for (int b = b0; b < std::min(n_blocks, b0 + kMaxProblems); ++b) {
      const GapBlock<double>& blk = blks[b];
      if (blk.n_rows == 0 || blk.n_cols == 0) continue;
      if (!blk.alpha) throw InvalidArgument("the GAP energy kernel needs weights");
      Problem& P = ps.p[ps.n++];
      kernel_problem(P, blk);
      P.alpha = blk.alpha + blk.col0;
      P.epart = energy ? part : nullptr;
      P.ldp = ld;
      P.wt = wts ? wts[b] : nullptr;
      P.ldw = gap_f64_k_stride(blk.n_cols);
      ps.normalize = blk.normalize;
      ps.zeta = blk.zeta;
      et.rows[et.n] = blk.row_idx;
      et.m[et.n] = blk.n_rows;
      et.tiles[et.n++] = gap_f64_energy_tiles(blk.n_cols);
    }
    launch<0>(ps, stream);
    if (energy) launch_energy_tiles(et, part, ld, energy, stream);
  }
}

void run_gap_f64_rows(const GapBlock<double>* blks, int n_blocks, double* out, int64_t ld, hipStream_t stream) {
  for (int b0 = 0; b0 < n_blocks; b0 += kMaxProblems) {
    ProblemSet ps{};
    for (int b = b0; b < std::min(n_blocks, b0 + kMaxProblems); ++b) {
      const GapBlock<double>& blk = blks[b];
      if (blk.n_rows == 0 || blk.n_cols == 0) continue;
      Problem& P = ps.p[ps.n++];
      kernel_problem(P, blk);
      P.G = out + blk.col0;
      P.ldg = ld;
      ps.normalize = blk.normalize;
      ps.zeta = blk.zeta;
    }
    launch<2>(ps, stream);
  }
}

void run_gram_f64(int64_t rows, int64_t n, const double* A, double* Ap, double* At, const int* iota, double* C,
                  hipStream_t stream) {
  if (rows == 0 || n == 0) return;
  if (n % 2 == 0) Ap = nullptr;  // (rows are 16-byte aligned as they are)
  const int64_t ldt = gap_f64_k_stride(rows);
  const dim3 grid(unsigned((n + 31) / 32), unsigned((rows + 31) / 32));
  RGPU_HIP(hipMemsetAsync(At, 0, sizeof(double) * size_t(n) * size_t(ldt), stream));
  hipLaunchKernelGGL(transpose_f64_kernel, grid, dim3(256), 0, stream, rows, n, A, At, ldt, Ap);
  RGPU_LAUNCH_CHECK();
  // C[i][:] = sum_r At[i][r] A[r][:], the force product with W~ = A^T
  ProblemSet ps{};
  ps.n = 1;
  Problem& P = ps.p[0];
  P.M = P.N = n;
  P.K = ldt;
  P.Kv = rows;
  P.A = At;
  P.lda = ldt;
  P.B = Ap ? Ap : A;
  P.ldb = Ap ? n + 1 : n;
  P.c_rows = iota;
  P.G = C;
  P.ldg = n;
  launch<1>(ps, stream);
}

void run_gap_f64_force(const GapBlock<double>* blks, int n_blocks, double* const* wts, const double* xg,
                       double xg_scale, double* G, hipStream_t stream) {
  for (int b0 = 0; b0 < n_blocks; b0 += kMaxProblems) {
    ProblemSet ps{};
    ps.xg_scale = xg_scale;
    for (int b = b0; b < std::min(n_blocks, b0 + kMaxProblems); ++b) {
      const GapBlock<double>& blk = blks[b];
      if (blk.n_rows == 0 || blk.n_cols == 0) continue;
      Problem& P = ps.p[ps.n++];
      P.M = blk.n_rows;
      P.N = blk.D;
      P.K = gap_f64_k_stride(blk.n_cols);
      P.Kv = blk.n_cols;
      P.A = wts[b];
      P.lda = P.K;
      P.a_rows = nullptr;
      P.B = blk.Tm + blk.col0 * blk.D;  // [K = sparse points][N = D]
      P.ldb = blk.D;
      P.c_rows = blk.row_idx;
      P.G = G;
      P.ldg = blk.D;
      P.xp = blk.normalize ? blk.X : nullptr;
      P.xg = xg;
      P.norm2 = blk.norm2;
    }
    launch<1>(ps, stream);
  }
}

}  // namespace rgpu
