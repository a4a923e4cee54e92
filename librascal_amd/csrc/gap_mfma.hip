// Mixed-precision GAP GEMMs on the gfx950 matrix cores.
//
// Both products of the GAP prediction are computed as C = A B^T with A and B
// stored row-major with the contraction index contiguous:
//   kernel:  K[r][m] = sum_d X[row(r)][d] T[col0+m][d]       (B = T, [M][D])
//   forces:  G[row(r)][d] = sum_m W~[r][m] T[col0+m][d]      (B = T^T, [D][M])
// Every operand arrives split into BF16 planes, x = hi + lo with
// hi = bf16(x), lo = bf16(x - hi) (the power spectrum and this kernel's own
// energy epilogue write them that way; the sparse points are split once at
// load time), so the main loop does no conversions: each algorithmic
// multiply-add is three v_mfma_f32_32x32x16_bf16 products (hi.hi + hi.lo +
// lo.hi) accumulated in FP32.
//
// Tiling: 256 threads (4 wavefronts, 2 x 2), block tile 128 x 128, K step 32;
// each wavefront owns 64 x 64 = 2 x 2 MFMA tiles (64 x 64 block tiles, one
// MFMA tile a wavefront, where there are few).  Two LDS stages (one
// barrier per K step), the next K step's global loads issued before the
// MFMAs of the current one.  Every operand row is 16-byte aligned and every
// K a multiple of 32: the packed feature rows are padded to that, and so are
// the sparse points of each species in the force product (W~ rows and T^T
// columns carry zero pads up to the next multiple of 32).  So the loads
// always go straight to LDS (global_load_lds_dwordx4) in a swizzled layout.
// Unpadded W~ went through a second, register-staged kernel with a guarded K
// tail: a whole prediction of 1331 centres against 2 x 1000 sparse points
// (n_max 10, l_max 8) took 572 us with it and takes 369 us with the pads.
// All species blocks of one
// product go in one grouped launch, dealt to the XCDs so that a row panel
// stays in one L2.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hh"
#include "gap_mfma.hh"
#include "packing.hh"

namespace rgpu {

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

constexpr int BM = 128, BN = 128, BK = 32, NT = 256;
constexpr int kMinBN = 64;  // of the smaller tiles
constexpr int kMaxProblems = 16;
constexpr int kGroupM = 8;  // row panels per tile group

__device__ __forceinline__ unsigned short bf16_bits(__bf16 h) {
  return __builtin_bit_cast(unsigned short, h);
}

struct Problem {
  int64_t M, N, K;             // C (M x N) = A (M x K) B (N x K)^T
  const unsigned short* Ahi;   // A rows, K contiguous
  const unsigned short* Alo;
  int64_t lda;
  const int* a_rows;           // gathered A rows (null: identity)
  const unsigned short* Bhi;   // B rows, K contiguous, already offset
  const unsigned short* Blo;
  int64_t ldb;
  const int* c_rows;           // output row ids (centre indices)
  int64_t tile0;               // first linear tile of this problem
  int tiles_m, tiles_n;        // tiles along M and N
  // kernel epilogue
  const double* norm2;
  const double* alpha;         // offset to the block's first sparse point
  double* epart;               // energy partials [tiles_n][ldp], by centre
  int64_t ldp;
  unsigned short* wth;         // [M][ldw] W~ split (may be null), columns N .. ldw zero
  unsigned short* wtl;
  int64_t ldw;
  // force epilogue
  float* G;
  int64_t ldg;
};

struct ProblemSet {
  Problem p[kMaxProblems];
  int64_t total_tiles;
  int n;
  int normalize;
  int zeta;
};

template <class T>
__device__ __forceinline__ T pow_int(T v, int n) {
  if (n == 0) return T(1);
  if (n == 1) return v;
  if (n == 2) return v * v;
  if (n == 3) return v * v * v;
  T r = T(1), x = v;
  unsigned u = unsigned(n);
  do {
    if (u & 1) r *= x;
    u >>= 1;
    x *= x;
  } while (u);
  return r;
}

// Epilogue of a TBM x TBN block tile whose wavefronts form 2 x 2 and own
// WI x WJ MFMA tiles each; esum: LDS [2][TBM]
template <int EPI, int TBM, int TBN, int WI, int WJ>
__device__ __forceinline__ void gemm_epilogue(const ProblemSet& ps, const Problem& P, int64_t r0,
                                              int64_t c0, f32x16 (&acc)[WI][WJ], double (*esum)[TBM]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // epilogue; element e = 4*g + q of a 32x32 tile sits at
  // row 8*g + 4*(lane/32) + q, column lane%32
  const int half = lane >> 5, fr = lane & 31;
  if (EPI == 0) {
    double rowsum[WI][16];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) rowsum[i][e] = 0.0;
#pragma unroll
    for (int i = 0; i < WI; ++i) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int rl = wm * 32 * WI + i * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
        const int64_t r = r0 + rl;
        if (r >= P.M) continue;
        const int centre = P.c_rows[r];
        double inv = 1.0;
        if (ps.normalize) {
          const double n2 = P.norm2[centre];
          inv = n2 > 0 ? 1.0 / sqrt(n2) : 1.0;
        }
#pragma unroll
        for (int j = 0; j < WJ; ++j) {
          const int64_t c = c0 + wn * 32 * WJ + j * 32 + fr;
          if (c >= P.N) {
            if (P.wth && c < P.ldw) P.wth[r * P.ldw + c] = P.wtl[r * P.ldw + c] = 0;
            continue;
          }
          const float k = float(double(acc[i][j][e]) * inv);
          const double a = P.alpha[c];
          rowsum[i][e] += a * double(pow_int(k, ps.zeta));
          if (P.wth) {
            const float g = ps.zeta > 1 ? float(ps.zeta) * pow_int(k, ps.zeta - 1) : 1.f;
            const float v = float(a) * g;
            const __bf16 h = (__bf16)v;
            P.wth[r * P.ldw + c] = bf16_bits(h);
            P.wtl[r * P.ldw + c] = bf16_bits((__bf16)(v - (float)h));
          }
        }
      }
    }
    // reduce over the 32 columns held by the lanes of each half
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        double v = rowsum[i][e];
        for (int off = 16; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        rowsum[i][e] = v;
      }
    if (fr == 0) {
#pragma unroll
      for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          esum[wn][wm * 32 * WI + i * 32 + 8 * (e >> 2) + 4 * half + (e & 3)] = rowsum[i][e];
    }
    __syncthreads();
    if (P.epart && tid < TBM) {
      const int64_t r = r0 + tid;
      if (r < P.M) P.epart[(c0 / TBN) * P.ldp + P.c_rows[r]] = esum[0][tid] + esum[1][tid];
    }
  } else {
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t r = r0 + wm * 32 * WI + i * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
        if (r >= P.M) continue;
        float* g = P.G + int64_t(P.c_rows[r]) * P.ldg;
#pragma unroll
        for (int j = 0; j < WJ; ++j) {
          const int64_t c = c0 + wn * 32 * WJ + j * 32 + fr;
          if (c < P.N) g[c] = acc[i][j][e];
        }
      }
  }
}

// s_waitcnt vmcnt(N) lgkmcnt(0) (gfx9 encoding)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}
// (__syncthreads would wait for every load in flight)
__device__ __forceinline__ void bare_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Direct-to-LDS variant (global_load_lds_dwordx4: the loads write LDS
// without passing through VGPRs).  A stage of one operand plane holds the
// tile's rows of one K step (BK = 32 values, 64 B) as groups of 16 rows, one
// wavefront load instruction (64 lanes x 16 B) per group; inside a group
// row r keeps its K quarter q (8 values) at slot 4 r + (q ^ dma_swz(r)), so
// that each instruction reads whole 64-byte row segments and the fragment
// reads (16 rows of one quarter per 16 lanes) hit distinct banks.
__device__ __forceinline__ int dma_swz(int r) { return (r ^ (r >> 2)) & 3; }
// slot of the fragment of lane l for 32-row block rb, 16-wide K chunk c
__device__ __forceinline__ int dma_frag_slot(int rb, int c, int l) {
  const int r = l & 15;
  return (2 * rb + ((l >> 4) & 1)) * 64 + 4 * r + ((2 * c + (l >> 5)) ^ dma_swz(r));
}

// LDS stages; three and four were no faster with either tile
constexpr int NS = 2;

template <int TBM, int TBN>
struct DmaLds {
  bf16x8 A[NS][2][TBM / 16 * 64];  // [stage][hi, lo][slot]
  bf16x8 B[NS][2][TBN / 16 * 64];
  double esum[2][TBM];
};

// TBM x TBN block tile of four wavefronts, NS LDS stages with NS - 1 K steps
// in flight; K % 32 == 0 and 16-byte aligned rows
template <int EPI, int TBM, int TBN>
__device__ __forceinline__ void gemm_tile_dma(const ProblemSet& ps, const Problem& P, int64_t r0,
                                              int64_t c0, DmaLds<TBM, TBN>& sm) {
  constexpr int W = NT / 64, WI = TBM / 64, WJ = TBN / 64;  // MFMA tiles of a wavefront
  constexpr int GA = TBM / 16 / W, GB = TBN / 16 / W;  // groups per plane and wavefront
  static_assert(GA * W * 16 == TBM && GB * W * 16 == TBN, "group partition");
  constexpr int PER = 2 * (GA + GB);  // load instructions per wavefront and K step
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // lane of a group load: row lane / 4, quarter q; rows past the matrix
  // edge repeat its last row (their results are never stored)
  const int rr = lane >> 2, q = (lane & 3) ^ dma_swz(rr);
  int64_t offa[GA], offb[GB];
#pragma unroll
  for (int j = 0; j < GA; ++j) {
    int64_t ra = r0 + (wave + W * j) * 16 + rr;
    ra = ra < P.M ? ra : P.M - 1;
    if (P.a_rows) ra = P.a_rows[ra];
    offa[j] = ra * P.lda + 8 * q;
  }
#pragma unroll
  for (int j = 0; j < GB; ++j) {
    int64_t rb = c0 + (wave + W * j) * 16 + rr;
    rb = rb < P.N ? rb : P.N - 1;
    offb[j] = rb * P.ldb + 8 * q;
  }
  const int64_t nk = P.K / BK;
  // loads of K step kt (clamped to the last one: the surplus loads at the
  // end land in stages that are never read) into stage s
  auto issue = [&](int s, int64_t kt) {
    const int64_t k = (kt < nk ? kt : nk - 1) * BK;
#pragma unroll
    for (int j = 0; j < GA; ++j) {
      const int g = (wave + W * j) * 64;
      __builtin_amdgcn_global_load_lds(P.Ahi + offa[j] + k, &sm.A[s][0][g], 16, 0, 0);
      __builtin_amdgcn_global_load_lds(P.Alo + offa[j] + k, &sm.A[s][1][g], 16, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < GB; ++j) {
      const int g = (wave + W * j) * 64;
      __builtin_amdgcn_global_load_lds(P.Bhi + offb[j] + k, &sm.B[s][0][g], 16, 0, 0);
      __builtin_amdgcn_global_load_lds(P.Blo + offb[j] + k, &sm.B[s][1][g], 16, 0, 0);
    }
  };

  f32x16 acc[WI][WJ];
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < WJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  auto compute = [&](int s) {
#pragma unroll
    for (int c = 0; c < BK / 16; ++c) {
      bf16x8 ah[WI], al[WI], bh[WJ], bl[WJ];
#pragma unroll
      for (int i = 0; i < WI; ++i) {
        const int f = dma_frag_slot(wm * WI + i, c, lane);
        ah[i] = sm.A[s][0][f];
        al[i] = sm.A[s][1][f];
      }
#pragma unroll
      for (int j = 0; j < WJ; ++j) {
        const int f = dma_frag_slot(wn * WJ + j, c, lane);
        bh[j] = sm.B[s][0][f];
        bl[j] = sm.B[s][1][f];
      }
#pragma unroll
      for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int j = 0; j < WJ; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
        }
    }
  };

#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s, s);
  int s_read = 0, s_fill = NS - 1;
  for (int64_t kt = 0; kt < nk; ++kt) {
    // this wavefront's loads of step kt are done once at most the NS - 2
    // later steps' remain; the barrier extends that to every wavefront and
    // orders the previous step's fragment reads before the refill of its
    // stage
    wait_vmcnt<(NS - 2) * PER>();
    bare_barrier();
    issue(s_fill, kt + NS - 1);
    compute(s_read);
    s_read = s_read + 1 == NS ? 0 : s_read + 1;
    s_fill = s_fill + 1 == NS ? 0 : s_fill + 1;
  }
  // no load may still write this workgroup's LDS when it exits
  wait_vmcnt<0>();
  gemm_epilogue<EPI, TBM, TBN, WI, WJ>(ps, P, r0, c0, acc, sm.esum);
}

// problem index and tile (row, column) of linear block bid.  Workgroups
// are dealt to the 8 XCDs round robin; each XCD takes a contiguous range of
// linear tiles, and the linear order walks groups of kGroupM row panels
// column by column, so the tiles resident on one XCD at a time form a
// square of row and column panels that share their operand panels through
// the XCD's L2.
__device__ __forceinline__ bool tile_of(const ProblemSet& ps, int* pi_out, int64_t* tm_out,
                                        int64_t* tn_out) {
  const int64_t per_xcd = (int64_t(gridDim.x) + 7) / 8;
  const int64_t bid = int64_t(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (bid >= ps.total_tiles) return false;
  int pi = 0;
  while (pi + 1 < ps.n && bid >= ps.p[pi + 1].tile0) ++pi;
  const Problem& P = ps.p[pi];
  const int64_t local = bid - P.tile0;
  const int64_t per_group = int64_t(kGroupM) * P.tiles_n;
  const int64_t grp = local / per_group, in = local - grp * per_group;
  const int64_t gm = std::min<int64_t>(kGroupM, P.tiles_m - grp * kGroupM);
  const int64_t tn = in / gm;
  *pi_out = pi;
  *tm_out = grp * kGroupM + (in - tn * gm);
  *tn_out = tn;
  return true;
}

// EPI 0: GAP kernel epilogue, 1: store rows of G
template <int EPI, int TBM, int TBN>
__global__ __launch_bounds__(NT, 2) void bf16x3_gemm_dma(ProblemSet ps) {
  int pi;
  int64_t tm, tn;
  if (!tile_of(ps, &pi, &tm, &tn)) return;
  const Problem& P = ps.p[pi];
  __shared__ __align__(16) DmaLds<TBM, TBN> sm;
  gemm_tile_dma<EPI, TBM, TBN>(ps, P, tm * TBM, tn * TBN, sm);
}

// Packed BF16 planes of the sparse points in both orientations: 32 points x
// 64 packed columns per workgroup, the values formed once (src: the one or
// two full-layout columns of a packed column, equal for a plain copy, -1 for
// a pad) and turned through LDS, so that both layouts are stored along their
// rows.  Memory bound; setting 4096 points of 14400 columns took 975 ms with
// the host loop it replaced and takes 178 ms, host copies of the values.
constexpr int kPrepM = 32, kPrepD = 64;
__global__ __launch_bounds__(NT) void split_sparse_kernel(const double* __restrict__ T, int64_t M, int64_t D,
                                                          int64_t Dq, const int2* __restrict__ src,
                                                          const int64_t* __restrict__ col, int64_t Mp,
                                                          unsigned short* __restrict__ t_hi,
                                                          unsigned short* __restrict__ t_lo,
                                                          unsigned short* __restrict__ tt_hi,
                                                          unsigned short* __restrict__ tt_lo) {
  __shared__ unsigned short th[kPrepD][kPrepM + 2], tl[kPrepD][kPrepM + 2];
  const int64_t d0 = int64_t(blockIdx.x) * kPrepD, m0 = int64_t(blockIdx.y) * kPrepM;
  const int dx = threadIdx.x & (kPrepD - 1), my = threadIdx.x / kPrepD;
  const int64_t d = d0 + dx;
  const int2 sc = d < Dq ? src[d] : make_int2(-1, -1);
  for (int k = my; k < kPrepM; k += NT / kPrepD) {
    const int64_t m = m0 + k;
    if (d >= Dq || m >= M) continue;
    const double* row = T + m * D;
    double v = 0.0;
    if (sc.x >= 0) v = sc.x == sc.y ? row[sc.x] : (row[sc.x] + row[sc.y]) * 0.70710678118654752440;
    const float x = float(v);
    const __bf16 h = (__bf16)x;
    const unsigned short hb = bf16_bits(h), lb = bf16_bits((__bf16)(x - (float)h));
    t_hi[m * Dq + d] = hb;
    t_lo[m * Dq + d] = lb;
    th[dx][k] = hb;
    tl[dx][k] = lb;
  }
  __syncthreads();
  const int mx = threadIdx.x & (kPrepM - 1), dy = threadIdx.x / kPrepM;
  const int64_t m = m0 + mx;
  const int64_t c = m < M ? col[m] : -1;
  if (c < 0) return;
  for (int k = dy; k < kPrepD && d0 + k < Dq; k += NT / kPrepM) {
    tt_hi[(d0 + k) * Mp + c] = th[k][mx];
    tt_lo[(d0 + k) * Mp + c] = tl[k][mx];
  }
}

// tile counts and first tiles of the set's problems for bm x bn tiles
int64_t layout_tiles(ProblemSet& ps, int bm, int bn) {
  int64_t tiles = 0;
  for (int i = 0; i < ps.n; ++i) {
    Problem& P = ps.p[i];
    P.tile0 = tiles;
    P.tiles_m = int((P.M + bm - 1) / bm);
    P.tiles_n = int((P.N + bn - 1) / bn);
    tiles += int64_t(P.tiles_m) * P.tiles_n;
  }
  return tiles;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Under three quarters of a 128 x 128 tile per CU, 64 x 64 tiles: a tile
// alone on its CU takes the same time however few there are (96 tiles, 60 K
// steps: 78 us, 48 us in small ones; 168 tiles, 208 K steps: 255 and 194 us),
// while with the chip full their extra operand traffic shows (512 tiles, 363 K
// steps: 602 and 1035 us).  They double the partial sums of the energies
// (rows x column tiles), which stay under 2^22 so that no batch outgrows a
// scratch array for it.
bool small_tiles(int64_t tiles, int64_t rows, int64_t cols) {
  return 4 * tiles <= 3 * int64_t(device_cu_count()) &&
         rows * ((cols + kMinBN - 1) / kMinBN) <= int64_t(1) << 22;
}

// columns per tile of the set's launch
template <int EPI>
int launch_set(ProblemSet& ps, hipStream_t stream) {
  if (ps.n == 0) return BN;
  for (int i = 0; i < ps.n; ++i) {
    const Problem& P = ps.p[i];
    if (P.K % BK != 0 || P.lda % 8 != 0 || P.ldb % 8 != 0 || !aligned16(P.Ahi) || !aligned16(P.Alo) ||
        !aligned16(P.Bhi) || !aligned16(P.Blo))
      throw InvalidArgument("internal: unaligned operands of the mixed GAP product");
  }
  auto go = [&](auto kern, int bm, int bn) {
    ps.total_tiles = layout_tiles(ps, bm, bn);
    if (ps.total_tiles == 0) return bn;
    const unsigned grid = unsigned((ps.total_tiles + 7) / 8 * 8);  // whole rounds over the 8 XCDs
    hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), 0, stream, ps);
    RGPU_LAUNCH_CHECK();
    return bn;
  };
  const int64_t tiles = layout_tiles(ps, BM, BN);
  int64_t cols = 0;
  for (int i = 0; i < ps.n; ++i) cols = std::max(cols, ps.p[i].N);
  if (EPI == 0 ? small_tiles(tiles, ps.p[0].ldp, cols) : small_tiles(tiles, 0, 0))
    return go(bf16x3_gemm_dma<EPI, 64, 64>, 64, 64);
  return go(bf16x3_gemm_dma<EPI, BM, BN>, BM, BN);
}

}  // namespace

bool mfma_available() { return true; }

void prepare_mixed_sparse(MixedSparse& ms, const double* T, int64_t M, int S, int N, int L1,
                          const std::vector<int64_t>& sp_off, hipStream_t stream) {
  // rows of T in the packed layout (packing.hh); a sparse point's diagonal
  // blocks need not be symmetric: (t[n1][n2] + t[n2][n1]) / sqrt 2 keeps
  // every product with a symmetric feature row exact
  const int K = S * (S + 1) / 2, KB = N * N * L1, KD = packed_diag_block(N, L1);
  const int64_t D = int64_t(K) * KB;
  const int64_t Dq = packed_row_stride(S, N, L1);  // zero pad columns
  ms.D = Dq;
  std::vector<int2> src(size_t(std::max<int64_t>(Dq, 1)), make_int2(-1, -1));
  for (int k = 0; k < K; ++k) {
    int a, b;
    key_pair(k, S, &a, &b);
    int2* dk = src.data() + packed_key_offset(a, b, S, N, L1);
    const int k0 = k * KB;
    for (int o = 0; o < (a < b ? KB : KD); ++o) {
      int n1 = 0, n2 = 0;
      const int l = o % L1;
      if (a == b) packed_pair(o / L1, N, &n1, &n2);
      dk[o] = a < b ? make_int2(k0 + o, k0 + o)
                    : make_int2(k0 + (n1 * N + n2) * L1 + l, k0 + (n2 * N + n1) * L1 + l);
    }
  }
  // columns of the force operand: the points of each batch species from a
  // multiple of 32 on, zero pads between (points of other species have none)
  ms.col.assign(size_t(S), 0);
  std::vector<int64_t> col(size_t(std::max<int64_t>(M, 1)), -1);
  ms.Mp = 0;
  for (int s = 0; s < S; ++s) {
    ms.col[size_t(s)] = ms.Mp;
    for (int64_t m = sp_off[size_t(s)]; m < sp_off[size_t(s) + 1]; ++m)
      col[size_t(m)] = ms.Mp + (m - sp_off[size_t(s)]);
    ms.Mp += gap_mixed_wt_stride(sp_off[size_t(s) + 1] - sp_off[size_t(s)]);
  }
  const size_t n = size_t(std::max<int64_t>(M * Dq, 1)), nt = size_t(std::max<int64_t>(ms.Mp * Dq, 1));
  unsigned short *th = ms.t_hi.reserve(n), *tl = ms.t_lo.reserve(n);
  unsigned short *tth = ms.tt_hi.reserve(nt), *ttl = ms.tt_lo.reserve(nt);
  RGPU_HIP(hipMemsetAsync(tth, 0, nt * 2, stream));
  RGPU_HIP(hipMemsetAsync(ttl, 0, nt * 2, stream));
  if (M > 0 && Dq > 0) {
    DeviceBuffer<int2> d_src;
    DeviceBuffer<int64_t> d_col;
    int2* ds = d_src.reserve(src.size());
    int64_t* dc = d_col.reserve(col.size());
    RGPU_HIP(hipMemcpyAsync(ds, src.data(), sizeof(int2) * src.size(), hipMemcpyHostToDevice, stream));
    RGPU_HIP(hipMemcpyAsync(dc, col.data(), sizeof(int64_t) * col.size(), hipMemcpyHostToDevice, stream));
    // column blocks along x: at most 65535 blocks of points along y at a time
    for (int64_t m0 = 0; m0 < M; m0 += int64_t(65535) * kPrepM) {
      const int64_t mm = std::min<int64_t>(M - m0, int64_t(65535) * kPrepM);
      hipLaunchKernelGGL(split_sparse_kernel,
                         dim3(unsigned((Dq + kPrepD - 1) / kPrepD), unsigned((mm + kPrepM - 1) / kPrepM)),
                         dim3(NT), 0, stream, T + m0 * D, mm, D, Dq, ds, dc + m0, ms.Mp, th + m0 * Dq,
                         tl + m0 * Dq, tth, ttl);
      RGPU_LAUNCH_CHECK();
    }
    RGPU_HIP(hipStreamSynchronize(stream));  // before the maps are freed
  }
}

int64_t gap_mixed_wt_stride(int64_t n_cols) { return (n_cols + BK - 1) / BK * BK; }

int gap_mixed_energy_tiles(const int64_t* rows, const int64_t* cols, int n_blocks, int64_t ld) {
  int64_t t = 0;
  for (int b0 = 0; b0 < n_blocks; b0 += kMaxProblems) {
    int64_t tiles = 0, widest = 0;
    for (int b = b0; b < std::min(n_blocks, b0 + kMaxProblems); ++b) {
      if (rows[b] == 0 || cols[b] == 0) continue;
      tiles += (rows[b] + BM - 1) / BM * ((cols[b] + BN - 1) / BN);
      widest = std::max(widest, cols[b]);
    }
    const int bn = small_tiles(tiles, ld, widest) ? kMinBN : BN;
    t = std::max(t, (widest + bn - 1) / bn);
  }
  return int(t);
}

void run_gap_mixed_kernel(const GapBlock<float>* blks, int n_blocks, const MixedSparse& ms,
                          SplitPlanes xs, double* energy, double* part, int64_t ld, const SplitPlanes* wts,
                          hipStream_t stream) {
  static_assert(kMaxProblems <= EnergyTiles::kMax, "one energy reduction per grouped launch");
  for (int b0 = 0; b0 < n_blocks; b0 += kMaxProblems) {
    ProblemSet ps{};
    EnergyTiles et;
    for (int b = b0; b < std::min(n_blocks, b0 + kMaxProblems); ++b) {
      const GapBlock<float>& blk = blks[b];
      if (blk.n_rows == 0 || blk.n_cols == 0) continue;
      Problem& P = ps.p[ps.n++];
      P.M = blk.n_rows;
      P.N = blk.n_cols;
      P.K = blk.D;
      P.Ahi = xs.hi;
      P.Alo = xs.lo;
      P.lda = blk.D;
      P.a_rows = blk.row_idx;
      P.Bhi = ms.t_hi.get() + blk.col0 * blk.D;
      P.Blo = ms.t_lo.get() + blk.col0 * blk.D;
      P.ldb = blk.D;
      P.c_rows = blk.row_idx;
      P.norm2 = blk.norm2;
      if (!blk.alpha) throw InvalidArgument("the GAP energy kernel needs weights");
      P.alpha = blk.alpha + blk.col0;
      P.epart = energy ? part : nullptr;
      P.ldp = ld;
      P.wth = wts ? wts[b].hi : nullptr;
      P.wtl = wts ? wts[b].lo : nullptr;
      P.ldw = gap_mixed_wt_stride(blk.n_cols);
      ps.normalize = blk.normalize;
      ps.zeta = blk.zeta;
      et.rows[et.n] = blk.row_idx;
      et.m[et.n] = blk.n_rows;
      et.n++;
    }
    const int bn = launch_set<0>(ps, stream);
    for (int i = 0; i < et.n; ++i) et.tiles[i] = int((ps.p[i].N + bn - 1) / bn);
    if (energy) launch_energy_tiles(et, part, ld, energy, stream);
  }
}

void run_gap_mixed_force(const GapBlock<float>* blks, int n_blocks, const MixedSparse& ms,
                         const SplitPlanes* wts, float* G, hipStream_t stream) {
  for (int b0 = 0; b0 < n_blocks; b0 += kMaxProblems) {
    ProblemSet ps{};
    for (int b = b0; b < std::min(n_blocks, b0 + kMaxProblems); ++b) {
      const GapBlock<float>& blk = blks[b];
      if (blk.n_rows == 0 || blk.n_cols == 0) continue;
      Problem& P = ps.p[ps.n++];
      P.M = blk.n_rows;
      P.N = blk.D;
      P.K = gap_mixed_wt_stride(blk.n_cols);  // zero pads on both operands
      P.Ahi = wts[b].hi;
      P.Alo = wts[b].lo;
      P.lda = P.K;
      P.a_rows = nullptr;
      P.Bhi = ms.tt_hi.get() + ms.col[size_t(b)];
      P.Blo = ms.tt_lo.get() + ms.col[size_t(b)];
      P.ldb = ms.Mp;
      P.c_rows = blk.row_idx;
      P.G = G;
      P.ldg = blk.D;
    }
    launch_set<1>(ps, stream);
  }
}

}  // namespace rgpu
