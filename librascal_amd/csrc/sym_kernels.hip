// Power spectrum in symmetric packed rows and its adjoint (sym_kernels.hh).
//
// The power spectrum multiplies tiles of C_l's rows on the FP64 matrix cores,
// both operands read from LDS in the same layout.  The adjoint walks one
// angular channel per wavefront with lane = row r of C_l, dL/dC_l[r][:] in
// registers; the row C_l[c][:] of every step is the same for the whole
// wavefront, so it is read through scalar loads and enters the FMAs as a
// scalar operand, beside one packed entry per step from LDS.  (A matrix-core
// form of that one took 354 us where this took 318, and takes 249 with several
// columns in flight: its operands come through the packed triangle, and it
// leaves fewer wavefronts in flight.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "common.hh"
#include "radial.hh"
#include "packing.hh"
#include "sym_kernels.hh"

namespace rgpu {

namespace {

constexpr int kThreads = 256, kWaves = kThreads / 64;

// constant address space: wavefront-uniform addresses become scalar loads
typedef const __attribute__((address_space(4))) double* uniform_ptr;

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__host__ __device__ constexpr int tri_i(int r) { return r * (r + 1) / 2; }

typedef double f64x4 __attribute__((ext_vector_type(4)));

// k-th of the units 0 .. n-1 (in descending order of work) of a wavefront, -1
// past the last: they are dealt to the nw wavefronts back and forth, which
// evens out the work (l_max 9, one channel a unit, 4 wavefronts: 27, 25, 24,
// 24 columns)
__device__ __forceinline__ int wave_unit(int n, int nw, int wave, int k) {
  const int u = nw * k + ((k & 1) ? nw - 1 - wave : wave);
  return u < n ? u : -1;
}

// the keys a <= b, a << 8 | b
__device__ __forceinline__ void key_table(int S, int* key_ab) {
  for (int k = threadIdx.x; k < S * (S + 1) / 2; k += kThreads) {
    int a, b;
    key_pair(k, S, &a, &b);
    key_ab[k] = (a << 8) | b;
  }
}

// f(std::integral_constant<int, l>) for the runtime l <= LM
template <int LM, class F>
__device__ __forceinline__ void with_channel(int l, F&& f) {
  if constexpr (LM >= 0) {
    if (l == LM)
      f(std::integral_constant<int, LM>{});
    else
      with_channel<LM - 1>(l, f);
  }
}

// One workgroup of eight wavefronts per centre, C in LDS (odd row stride: no
// bank conflicts); a unit is a 16 x 16 tile (rows of C_l against rows of C_l, on
// and above the diagonal) of one channel on the matrix cores (16x16x4: a lane
// holds A[lane % 16][lane / 16], B[lane / 16][lane % 16] and the rows lane / 16 + 4 e
// of column lane % 16 of the result), the lanes of a column run along the
// packed entries of c.  Memory bound for many centres: 4096 centres of 4
// species, n_max 12, l_max 9 223 -> 132 us (0.54 GB), 4689 of n_max 8, l_max 6
// 70 -> 44 us, 1024 of 2 species, n_max 10, l_max 8 18.8 -> 14.5 us, against a
// lane per row and FMAs with the other row as a scalar operand, whose loads'
// latency bound it.
constexpr int kPowerWaves = 8;
__global__ __launch_bounds__(64 * kPowerWaves) void sym_power_kernel(int R, int L, int64_t ld,
                                                                     const double* __restrict__ c,
                                                                     double* __restrict__ p,
                                                                     double* __restrict__ norm2) {
  const int64_t i = blockIdx.x;
  const int LL = (L + 1) * (L + 1), LS = LL | 1, TRI = tri_i(R);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  extern __shared__ __align__(64) unsigned char smem_raw[];
  double* cs = reinterpret_cast<double*>(smem_raw);
  __shared__ double red[kPowerWaves];
  const double* ci = c + i * int64_t(R) * LL;
  for (int r = wave; r < R; r += kPowerWaves)
    for (int k = lane; k < LL; k += 64) cs[r * LS + k] = ci[r * LL + k];
  __syncthreads();
  double ss = 0.0;
  const int q = lane >> 4, x = lane & 15, RT = (R + 15) / 16, pairs = RT * (RT + 1) / 2;
  for (int k = wave; k < (L + 1) * pairs; k += kPowerWaves) {
    const int l = L - k / pairs, u = k - (L - l) * pairs, M = 2 * l + 1;
    const double f = 1.0 / sqrt(double(M)), f2 = f * 1.41421356237309504880;
    double* out = p + i * ld + int64_t(l) * TRI;
    int ct = 0;
    while (tri_i(ct + 1) <= u) ++ct;
    const int rt = u - tri_i(ct);
    const double* a = cs + min(16 * ct + x, R - 1) * LS + l * l + q;
    const double* b = cs + min(16 * rt + x, R - 1) * LS + l * l + q;
    f64x4 acc = {0, 0, 0, 0};
    for (int m = 0; m < M; m += 4) {
      const bool in = m + q < M;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? a[m] : 0.0, in ? b[m] : 0.0, acc, 0, 0, 0);
    }
    const int row = 16 * rt + x;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int col = 16 * ct + q + 4 * e;
      if (row <= col && col < R) {
        const double v = acc[e] * (row < col ? f2 : f);
        out[tri_i(col) + row] = v;
        ss += v * v;
      }
    }
  }
  for (int64_t o = int64_t(L + 1) * TRI + threadIdx.x; o < ld; o += 64 * kPowerWaves) p[i * ld + o] = 0.0;
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_down(ss, off, 64);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kPowerWaves; ++w) t += red[w];
    norm2[i] = t;
  }
}

// Rows [r0, r0 + 64) (a lane each) and orders of group grp of GM of one channel
// of the product below: dc (dL/dc of the centre) rows lm of channel l from the
// packed triangle w, with its diagonal times sqrt 2 in LDS, or (kMemory) as it is
// in memory, alpha w - beta p (p may be null).
template <int LM, int GM, bool kMemory>
__device__ __forceinline__ void contract_channel(int ll, int r0, int grp, int R, int N, int LL, int lane,
                                                 const double* w, const double* p, double alpha, double beta,
                                                 const double* ci, double* __restrict__ dc) {
  const double rt2 = 1.41421356237309504880;
  with_channel<LM>(ll, [&](auto lc) {
    constexpr int l = decltype(lc)::value, M = 2 * l + 1, CNT = (M + GM - 1) / GM;
    const int m_own = grp * CNT;
    if (m_own >= M) return;
    // (the last group may overlap the one before; it stores its own orders)
    const int m0 = GM == 1 ? 0 : min(m_own, M - CNT);
    const double f = rt2 / sqrt(double(M));
    const int r = min(r0 + lane, R - 1);
    double acc[CNT];
#pragma unroll
    for (int m = 0; m < CNT; ++m) acc[m] = 0.0;
    uniform_ptr y = (uniform_ptr)(ci + l * l + m0);
    int a = tri_i(r);
    // (columns whose scalar loads are in flight together, by the registers)
    constexpr int U = CNT <= 4 ? 8 : (CNT <= 9 ? 4 : (CNT <= 19 ? 2 : 1));
#pragma unroll U
    for (int col = 0; col < R; ++col, y += LL) {
      double v;
      if constexpr (kMemory) {
        v = p ? alpha * w[a] - beta * p[a] : w[a];
        v *= col == r ? rt2 : 1.0;
      } else {
        v = w[a];
      }
      a += col < r ? 1 : col + 1;
#pragma unroll
      for (int m = 0; m < CNT; ++m) acc[m] += v * y[m];
    }
    if (r0 + lane < R) {
      const int s = r / N, n = r - s * N;
      double* o = dc + int64_t(s) * LL * N + n;
#pragma unroll
      for (int m = 0; m < CNT; ++m)
        if (GM == 1 || m0 + m >= m_own) o[(l * l + m0 + m) * N] = f * acc[m];
    }
  });
}

// dL/dC_l[r][m] = f_l sqrt 2 sum_c w(r, c) C_l[c][m], w the packed entry
// dL/dp(r, c) (times sqrt 2 on the diagonal).  The channel's triangle of
// dL/dp is formed in LDS, straight in its packed order; a lane's walk along its
// row, tri(r) + c up to the diagonal and tri(c) + r after it, is free of bank
// conflicts there (triangular numbers run through every residue of a power of
// two).
//
// With p the packed rows G hold dL/dX of X = p / |p| and dL/dp = G / |p| - x p /
// |p|^2 is made on the way, x = xg[i], or (xg null) the n_dot values of the
// centre's products p . G that packing left in dot, over |p|.
//
// kShare: kOwn a triangle for each wavefront, which takes whole channels;
// kShared one for the workgroup, whose wavefronts take blocks of 64 rows and
// GM groups of the orders; kNone the entries gathered from memory (the triangle
// too large for the LDS).
//
// Bound by the memory it streams and the latency of the scalar loads, which the
// unrolled columns take together: 4096 centres, 4 species, n_max 12, l_max 9:
// 0.25 ms for 0.93 GB (0.32 one column at a time), where the key contraction
// of the fused FP64 adjoint it replaced took about 1.0 ms.
enum { kOwn, kShared, kNone };

template <int LM, int kShare, int GM, bool kProject>
__global__ __launch_bounds__(kThreads) void sym_contract_kernel(int R, int N, int L, int64_t ld,
                                                                const double* __restrict__ c,
                                                                const double* __restrict__ p,
                                                                const double* __restrict__ norm2,
                                                                const double* __restrict__ xg,
                                                                const double* __restrict__ dot, int n_dot,
                                                                const double* __restrict__ G,
                                                                double* __restrict__ dc) {
  const int64_t i = blockIdx.x;
  const int L1 = L + 1, LL = L1 * L1, TRI = tri_i(R);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double rt2 = 1.41421356237309504880;
  extern __shared__ __align__(64) unsigned char smem_raw[];
  double* W = reinterpret_cast<double*>(smem_raw) + (kShare == kOwn ? wave * TRI : 0);
  const double* Gi = G + i * ld;
  const double* pi = kProject ? p + i * ld : nullptr;
  double alpha = 1.0, beta = 0.0;
  if constexpr (kProject) {
    const double n2 = norm2[i];
    if (n2 > 0) {
      double x = 0.0;
      if (xg) {
        x = xg[i];
      } else {
        for (int k = 0; k < n_dot; ++k) x += dot[i * n_dot + k];
        x /= sqrt(n2);
      }
      alpha = 1.0 / sqrt(n2);
      beta = x / n2;
    }
  }
  const double* ci = c + i * int64_t(R) * LL;
  double* di = dc + i * int64_t(R) * LL;
  if constexpr (kShare == kOwn) {
    for (int k = 0; k * kWaves <= L; ++k) {
      const int u = wave_unit(L1, kWaves, wave, k), lk = L - u;
      if (u < 0) continue;
      const double *g = Gi + lk * TRI, *q = kProject ? pi + lk * TRI : nullptr;
      wave_sync();  // the previous channel is read
      // (many loads in flight: the runs come from memory)
#pragma unroll 16
      for (int t = lane; t < TRI; t += 64) W[t] = kProject ? alpha * g[t] - beta * q[t] : g[t];
      wave_sync();
      for (int r = lane; r < R; r += 64) W[tri_i(r) + r] *= rt2;
      wave_sync();
      for (int rb = 0; rb < R; rb += 64)
        contract_channel<LM, 1, false>(lk, rb, 0, R, N, LL, lane, W, nullptr, 1.0, 0.0, ci, di);
    }
  } else {
    const int RB = (R + 63) / 64;
    for (int l = L - int(blockIdx.y); l >= 0; l -= int(gridDim.y)) {
      const double *g = Gi + l * TRI, *q = kProject ? pi + l * TRI : nullptr;
      if constexpr (kShare == kShared) {
        __syncthreads();  // the previous channel is read
#pragma unroll 8
        for (int t = threadIdx.x; t < TRI; t += kThreads) W[t] = kProject ? alpha * g[t] - beta * q[t] : g[t];
        __syncthreads();
        for (int r = threadIdx.x; r < R; r += kThreads) W[tri_i(r) + r] *= rt2;
        __syncthreads();
      }
      for (int u = wave; u < RB * GM; u += kWaves)
        contract_channel<LM, GM, kShare == kNone>(l, (u / GM) * 64, u % GM, R, N, LL, lane, kShare == kNone ? g : W, q,
                                                  alpha, beta, ci, di);
    }
  }
}

// The same from full rows of dL/dX, the whole packed row formed in LDS first
// (channels LT apart): the full row is read once along itself, and no packed row
// goes through memory.  4689 centres of 4 species, n_max 8, l_max 6: 173 us,
// bound by the chain of its phases.
__host__ __device__ inline int full_stride(int R) { return tri_i(R) | 1; }

template <int LM>
__global__ __launch_bounds__(kThreads) void sym_contract_full_kernel(int R, int N, int L, int64_t ld,
                                                                     const double* __restrict__ c,
                                                                     const double* __restrict__ p,
                                                                     const double* __restrict__ norm2,
                                                                     const double* __restrict__ G,
                                                                     double* __restrict__ dc) {
  const int64_t i = blockIdx.x;
  const int L1 = L + 1, LL = L1 * L1, TRI = tri_i(R), LT = full_stride(R), S = R / N, NL = N * L1, KB = N * NL;
  const int K = S * (S + 1) / 2;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double rt2 = 1.41421356237309504880;
  extern __shared__ __align__(64) unsigned char smem_raw[];
  double* W = reinterpret_cast<double*>(smem_raw);
  int* key_ab = reinterpret_cast<int*>(W + L1 * LT);
  __shared__ double red[kWaves];
  key_table(S, key_ab);
  __syncthreads();
  const double* Gi = G + i * int64_t(K) * KB;
  const float inv_kb = 1.0f / float(KB), inv_nl = 1.0f / float(NL), inv_l = 1.0f / float(L1);
  // (several loads in flight, then the mirrors of the diagonal keys' entries)
  constexpr int U = 8;
  for (int e0 = threadIdx.x; e0 < K * KB; e0 += U * kThreads) {
    double v[U], w[U];
    int to[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = Gi[min(e0 + u * kThreads, K * KB - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = min(e0 + u * kThreads, K * KB - 1);
      int k = int((float(e) + 0.5f) * inv_kb);
      k -= k * KB > e ? 1 : 0;
      k += (k + 1) * KB <= e ? 1 : 0;
      const int o = e - k * KB, n1 = int((float(o) + 0.5f) * inv_nl), o1 = o - n1 * NL;
      const int n2 = int((float(o1) + 0.5f) * inv_l), l = o1 - n2 * L1;
      const int a = key_ab[k] >> 8, b = key_ab[k] & 255;
      to[u] = a == b && n1 > n2 ? -1 : l * LT + tri_i(b * N + n2) + a * N + n1;
      if (a == b && n1 < n2) {
        w[u] = Gi[k * KB + n2 * NL + n1 * L1 + l];
        v[u] *= 0.70710678118654752440;
      } else {
        w[u] = 0.0;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (to[u] >= 0) W[to[u]] = v[u] + 0.70710678118654752440 * w[u];
  }
  __syncthreads();
  if (p) {
    const double n2 = norm2[i];
    const double* pi = p + i * ld;
    const float inv_t = 1.0f / float(TRI);
    auto channel_of = [&](int t) { return int((float(t) + 0.5f) * inv_t); };
    double d = 0.0;
#pragma unroll 8
    for (int t = threadIdx.x; t < L1 * TRI; t += kThreads) d += pi[t] * W[t + channel_of(t) * (LT - TRI)];
    for (int off = 32; off > 0; off >>= 1) d += __shfl_down(d, off, 64);
    if (lane == 0) red[wave] = d;
    __syncthreads();
    if (n2 > 0) {
      const double x = ((red[0] + red[1]) + (red[2] + red[3])) / sqrt(n2);
      const double alpha = 1.0 / sqrt(n2), beta = x / n2;
#pragma unroll 8
      for (int t = threadIdx.x; t < L1 * TRI; t += kThreads) {
        double* w = W + t + channel_of(t) * (LT - TRI);
        *w = alpha * *w - beta * pi[t];
      }
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < L1 * R; e += kThreads) {
    const int l = e / R, r = e - l * R;
    W[l * LT + tri_i(r) + r] *= rt2;
  }
  __syncthreads();
  for (int k = 0; k * kWaves <= L; ++k) {
    const int u = wave_unit(L1, kWaves, wave, k);
    if (u < 0) continue;
    for (int rb = 0; rb < R; rb += 64)
      contract_channel<LM, 1, false>(L - u, rb, 0, R, N, LL, lane, W + (L - u) * LT, nullptr, 1.0, 0.0,
                                     c + i * int64_t(R) * LL, dc + i * int64_t(R) * LL);
  }
}

// dL/dc of several sparse points (sets) at kSetCentres centres of their
// species, one workgroup for a set: with W the symmetric matrix of a packed
// channel, dL/dC_l = alpha f W(T) C_l - beta f W(p) C_l, whose second product
// E does not depend on the set and comes from memory.  The columns of C_l of
// all the centres side by side make the first a matrix product without
// padding (16x16x4: a lane holds A[lane % 16][lane / 16], B[lane / 16][lane % 16]
// and the rows lane / 16 + 4 e of column lane % 16 of the result); T's channel is
// staged once in LDS (from memory where it is too large).  Forming alpha T -
// beta p for each centre and set read both rows for every one of them and
// took 1.18 ms for 300 sets of 983 centres in three species (n_max 8, l_max
// 6); this takes 0.89 ms, bound by the gathered 8-byte loads of c and E and
// the stores (W as a full matrix in LDS, with fewer index operations: 0.98).
constexpr int kSetCentres = 16;

template <bool LDS>
__global__ __launch_bounds__(kThreads) void sym_contract_sets_kernel(int R, int N, int L, int64_t ld, SymSets sets,
                                                                     const double* __restrict__ c,
                                                                     const double* __restrict__ norm2,
                                                                     const double* __restrict__ E,
                                                                     const double* __restrict__ T,
                                                                     double* __restrict__ dc) {
  const int L1 = L + 1, LL = L1 * L1, TRI = tri_i(R), S = R / N;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = lane >> 4, x = lane & 15;
  const int64_t set = blockIdx.y, i0 = int64_t(blockIdx.x) * kSetCentres;
  const int nc = int(min(int64_t(kSetCentres), sets.n_ids - i0));
  const double rt2 = 1.41421356237309504880;
  extern __shared__ __align__(64) unsigned char smem_raw[];
  double* W = reinterpret_cast<double*>(smem_raw);
  __shared__ double al[kSetCentres], be[kSetCentres];
  __shared__ int centre[kSetCentres];
  if (threadIdx.x < kSetCentres) {
    // dL/dX = zeta d^(zeta - 1) T, d = X . T (a centre past the end: unused)
    const int i = sets.ids[i0 + min(int(threadIdx.x), nc - 1)];
    const double d = sets.dot[i * sets.ld_dot + set];
    double a = double(sets.zeta), b = 0.0;
    for (int k = 1; k < sets.zeta; ++k) a *= d;
    if (E) {
      const double n2 = norm2[i];
      if (n2 > 0) {
        b = a * d / n2;
        a /= sqrt(n2);
      }
    }
    centre[threadIdx.x] = i;
    al[threadIdx.x] = a;
    be[threadIdx.x] = b;
  }
  const double* Ts = T + set * ld;
  const int B = S * LL * N;
  double* dcs = dc + (set * sets.n_ids + i0) * B;
  const float inv_n = 1.0f / float(N);
  for (int l = L - int(blockIdx.z); l >= 0; l -= int(gridDim.z)) {
    const int M = 2 * l + 1, cols = nc * M;
    const double f = rt2 / sqrt(double(M));
    const double* g = Ts + l * TRI;
    if constexpr (LDS) {
      __syncthreads();  // the previous channel is read
#pragma unroll 4
      for (int t = threadIdx.x; t < TRI; t += kThreads) W[t] = g[t];
      __syncthreads();
      for (int r = threadIdx.x; r < R; r += kThreads) W[tri_i(r) + r] *= rt2;
    }
    __syncthreads();
    const float inv_m = 1.0f / float(M);
    auto centre_of = [&](int col) { return int((float(col) + 0.5f) * inv_m); };
    for (int c0 = 16 * wave; c0 < cols; c0 += 16 * kWaves) {
      const int col = min(c0 + x, cols - 1), ic = centre_of(col);
      const double* cp = c + int64_t(centre[ic] * R) * LL + l * l + (col - ic * M);
      // this lane's four columns of the result
      const double* ee[4];
      double* oo[4];
      double av[4], bv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int oc = min(c0 + q + 4 * e, cols - 1), io = centre_of(oc), o = (l * l + (oc - io * M)) * N;
        ee[e] = E + (E ? int64_t(centre[io]) * B + o : 0);
        oo[e] = dcs + int64_t(io) * B + o;
        av[e] = al[io] * f;
        bv[e] = be[io];
      }
      for (int rb = 0; rb < R; rb += 16) {
        const int r = min(rb + x, R - 1), tr = tri_i(r);
        const int s = int((float(r) + 0.5f) * inv_n), sn = s * LL * N + (r - s * N);
        double ev[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) ev[e] = E ? ee[e][sn] : 0.0;
        f64x4 acc = {0, 0, 0, 0};
        // (rows past R: a zero operand)
#pragma unroll 6
        for (int k0 = 0; k0 < R; k0 += 4) {
          const int k = min(k0 + q, R - 1), t = k <= r ? tr + k : tri_i(k) + r;
          const double w = LDS ? W[t] : g[t] * (k == r ? rt2 : 1.0);
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(k0 + q < R ? cp[k * LL] : 0.0, k0 + q < R ? w : 0.0, acc, 0, 0, 0);
        }
        if (rb + x < R) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c0 + q + 4 * e < cols) oo[e][sn] = av[e] * acc[e] - bv[e] * ev[e];
        }
      }
    }
  }
}

// Full row <-> symmetric packed row, KC key blocks at a time through LDS
// ([key][n1][n2][l] with an odd n1 stride): both sides move along their rows
// (whole key blocks, runs of N packed entries), and several keys per pass keep
// enough loads in flight.  The passes of a row go to gridDim.y workgroups, more
// than one where there are few rows.  Memory bound.
// kExtra: kCheck *flag = 1 when a diagonal key's block of some row is not
// symmetric (every writer stores the same value); kDot dot[i gridDim.y + y] =
// this workgroup's part of p . G.
enum { kPlain, kCheck, kDot };
template <int kExtra>
__global__ __launch_bounds__(kThreads) void sym_pack_kernel(int S, int N, int L1, int KC, int64_t ld,
                                                            const double* __restrict__ full,
                                                            const int64_t* __restrict__ rows,
                                                            double* __restrict__ out, int* __restrict__ flag,
                                                            const double* __restrict__ p, double* __restrict__ dot) {
  const int64_t i = blockIdx.x;
  bool differ = false;
  double sum = 0.0;
  const int K = S * (S + 1) / 2, NL = N * L1, KB = N * NL, NS = NL | 1, TRI = tri_i(S * N), NN = N * N;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  extern __shared__ __align__(64) unsigned char smem_raw[];
  double* b = reinterpret_cast<double*>(smem_raw);
  int* key_ab = reinterpret_cast<int*>(b + size_t(KC) * N * NS);
  const double* src = full + (rows ? rows[i] : i) * (int64_t(K) * KB);
  double* dst = out + i * ld;
  const double* pi = kExtra == kDot ? p + i * ld : nullptr;
  const float inv_nl = 1.0f / float(NL);
  key_table(S, key_ab);
  for (int k0 = int(blockIdx.y) * KC; k0 < K; k0 += int(gridDim.y) * KC) {
    const int kc = min(KC, K - k0);
    __syncthreads();
#pragma unroll 8
    for (int e = threadIdx.x; e < kc * KB; e += kThreads) {
      const int r = int((float(e) + 0.5f) * inv_nl);
      b[r * (NS - NL) + e] = src[int64_t(k0) * KB + e];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kc * NN; t += kThreads) {
      const int kk = t / NN, tt = t - kk * NN, n2 = tt / N, n1 = tt - n2 * N;
      const int sa = key_ab[k0 + kk] >> 8, sb = key_ab[k0 + kk] & 255;
      if (sa == sb && n1 > n2) continue;
      const bool sym = sa == sb && n1 < n2;
      const double *bk = b + kk * N * NS, *b0 = bk + n1 * NS + n2 * L1, *b1 = bk + n2 * NS + n1 * L1;
      int64_t o = tri_i(sb * N + n2) + sa * N + n1;
#pragma unroll 4
      for (int l = 0; l < L1; ++l, o += TRI) {
        const double v = sym ? (b0[l] + b1[l]) * 0.70710678118654752440 : b0[l];
        dst[o] = v;
        if (kExtra == kCheck && sym) differ |= b0[l] != b1[l];
        if (kExtra == kDot) sum += v * pi[o];
      }
    }
  }
  if (blockIdx.y == 0)
    for (int64_t o = int64_t(L1) * TRI + threadIdx.x; o < ld; o += kThreads) dst[o] = 0.0;
  if (kExtra == kCheck && differ) *flag = 1;
  if constexpr (kExtra == kDot) {
    __shared__ double red[kWaves];
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) dot[i * gridDim.y + blockIdx.y] = (red[0] + red[1]) + (red[2] + red[3]);
  }
}

__global__ __launch_bounds__(kThreads) void sym_unpack_kernel(int S, int N, int L1, int KC, int64_t ld,
                                                              const double* __restrict__ p,
                                                              const int64_t* __restrict__ rows,
                                                              const double* __restrict__ norm2, int normalize,
                                                              double* __restrict__ out) {
  const int64_t i = rows ? rows[blockIdx.x] : int64_t(blockIdx.x);
  const int K = S * (S + 1) / 2, NL = N * L1, KB = N * NL, NS = NL | 1, TRI = tri_i(S * N), NN = N * N;
  extern __shared__ __align__(64) unsigned char smem_raw[];
  double* b = reinterpret_cast<double*>(smem_raw);
  int* key_ab = reinterpret_cast<int*>(b + size_t(KC) * N * NS);
  const double* src = p + i * ld;
  double* dst = out + int64_t(blockIdx.x) * (int64_t(K) * KB);
  const float inv_nl = 1.0f / float(NL);
  key_table(S, key_ab);
  double nr = 1.0;
  if (normalize && norm2[i] > 0) nr = sqrt(norm2[i]);
  for (int k0 = int(blockIdx.y) * KC; k0 < K; k0 += int(gridDim.y) * KC) {
    const int kc = min(KC, K - k0);
    __syncthreads();
    for (int t = threadIdx.x; t < kc * NN; t += kThreads) {
      const int kk = t / NN, tt = t - kk * NN, n2 = tt / N, n1 = tt - n2 * N;
      const int sa = key_ab[k0 + kk] >> 8, sb = key_ab[k0 + kk] & 255;
      if (sa == sb && n1 > n2) continue;
      const bool sym = sa == sb && n1 < n2;
      double *bk = b + kk * N * NS, *b0 = bk + n1 * NS + n2 * L1, *b1 = bk + n2 * NS + n1 * L1;
      const double* q = src + tri_i(sb * N + n2) + sa * N + n1;
#pragma unroll 4
      for (int l = 0; l < L1; ++l, q += TRI) {
        double v = *q;
        if (sym) {
          v *= 0.70710678118654752440;
          b1[l] = v;
        }
        b0[l] = v;
      }
    }
    __syncthreads();
#pragma unroll 4
    for (int e = threadIdx.x; e < kc * KB; e += kThreads) {
      const int r = int((float(e) + 0.5f) * inv_nl);
      dst[int64_t(k0) * KB + e] = b[r * (NS - NL) + e] / nr;
    }
  }
}

template <class K>
void allow_lds(K kernel, size_t smem) {
  if (smem > 160 * 1024)
    throw InvalidArgument("hypers need " + std::to_string(smem) +
                          " bytes of LDS per workgroup, more than the device provides");
  if (smem > 64 * 1024)
    RGPU_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(smem)));
}

// key blocks per pass of the row conversions (four workgroups per CU, one
// block at least) and their LDS
int key_blocks(int S, int N, int L1) {
  const size_t kb = sizeof(double) * size_t(N) * ((N * L1) | 1);
  return std::max(1, std::min(S * (S + 1) / 2, int(36 * 1024 / kb)));
}
size_t key_lds(int S, int N, int L1) {
  return sizeof(double) * size_t(key_blocks(S, N, L1)) * N * ((N * L1) | 1) + sizeof(int) * size_t(S * (S + 1) / 2);
}

}  // namespace

void launch_sym_power(int S, int N, int L1, int64_t n, const double* c, double* p, double* norm2,
                      hipStream_t stream) {
  if (n == 0) return;
  const int R = S * N;
  const size_t smem = sizeof(double) * size_t(R) * ((L1 * L1) | 1);
  allow_lds(sym_power_kernel, smem);
  hipLaunchKernelGGL(sym_power_kernel, dim3(unsigned(n)), dim3(64 * kPowerWaves), smem, stream, R, L1 - 1,
                     sym_row_stride(S, N, L1), c, p, norm2);
  RGPU_LAUNCH_CHECK();
}

namespace {

constexpr size_t kContractLds = 156 * 1024;
// sym_contract_full_kernel: two workgroups per CU at least.  Adjoint from full
// rows, whole in LDS against packed first: 2000 centres of 2 species, n_max 12,
// l_max 9 (23 KB) 129 and 158 us, 3 species (52 KB) 237 and 303, 4 species, n_max
// 10, l_max 8 (57 KB) 261 and 310, 1500 of 6, n_max 8, l_max 6 (64 KB) 147 and 225,
// but 2000 of 4, n_max 12, l_max 9 (91 KB) 509 and 441.
constexpr size_t kFullLds = 78 * 1024;
// A triangle for each wavefront while two workgroups per CU have them (R <= 65),
// else one for the workgroup, four times as many of which fit.  Adjoint of a
// prediction, own against shared: 64 rows (8 species, n_max 8, l_max 4) 76 and
// 85 us, 52 rows (4, 13, 8) 235 and 321; 72 rows (6, 12, 9) 383 and 265, 90 rows
// (10, 9, 4) 353 and 248 (1000 to 2000 centres).
constexpr size_t kOwnLds = 68 * 1024;

// workgroups that share a row's passes in the row conversions: one but where
// there are too few rows to fill the chip
unsigned row_split(int S, int N, int L1, int64_t n) {
  const int kc = key_blocks(S, N, L1), passes = (S * (S + 1) / 2 + kc - 1) / kc;
  return unsigned(std::max<int64_t>(1, std::min<int64_t>(passes, 1024 / n)));
}

template <int kExtra>
void go_pack(int S, int N, int L1, int64_t n, unsigned split, const double* full, const int64_t* rows, double* out,
             int* flag, const double* p, double* dot, hipStream_t stream) {
  const size_t smem = key_lds(S, N, L1);
  allow_lds(sym_pack_kernel<kExtra>, smem);
  hipLaunchKernelGGL(sym_pack_kernel<kExtra>, dim3(unsigned(n), split), dim3(kThreads), smem, stream, S, N, L1,
                     key_blocks(S, N, L1), sym_row_stride(S, N, L1), full, rows, out, flag, p, dot);
  RGPU_LAUNCH_CHECK();
}

template <bool kProject>
void go_contract(int S, int N, int L1, int64_t n, const double* c, const double* p, const double* norm2,
                 const double* xg, const double* dot, int n_dot, const double* G, double* dc, hipStream_t stream) {
  const int R = S * N;
  const size_t tri = sizeof(double) * size_t(sym_tri(R));
  auto go = [&](auto kern, size_t smem, unsigned split) {
    allow_lds(kern, smem);
    hipLaunchKernelGGL(kern, dim3(unsigned(n), split), dim3(kThreads), smem, stream, R, N, L1 - 1,
                       sym_row_stride(S, N, L1), c, p, norm2, xg, dot, n_dot, G, dc);
    RGPU_LAUNCH_CHECK();
  };
  auto by_form = [&](auto lm) {
    constexpr int LM = decltype(lm)::value;
    // (channels over more workgroups where there are few centres)
    const unsigned split = unsigned(std::max<int64_t>(1, std::min<int64_t>(L1, 1024 / n)));
    const int rb = (R + 63) / 64;
    if (kWaves * tri <= kOwnLds)
      go(sym_contract_kernel<LM, kOwn, 1, kProject>, kWaves * tri, 1);
    else if (tri > kContractLds)
      go(sym_contract_kernel<LM, kNone, 2, kProject>, 0, split);
    else if (rb == 1 || rb == 3)
      go(sym_contract_kernel<LM, kShared, 4, kProject>, tri, split);
    else
      go(sym_contract_kernel<LM, kShared, 2, kProject>, tri, split);
  };
  if (L1 <= 10)
    by_form(std::integral_constant<int, 9>{});
  else
    by_form(std::integral_constant<int, kMaxL1 - 1>{});
}

}  // namespace

void launch_sym_contract(int S, int N, int L1, int64_t n, const double* c, const double* G, double* dc,
                         hipStream_t stream) {
  if (n == 0) return;
  go_contract<false>(S, N, L1, n, c, nullptr, nullptr, nullptr, nullptr, 0, G, dc, stream);
}

void launch_sym_contract_projected(int S, int N, int L1, int64_t n, const double* c, const double* p,
                                   const double* norm2, const double* xg, const double* G, double* dc,
                                   hipStream_t stream) {
  if (n == 0) return;
  go_contract<true>(S, N, L1, n, c, p, norm2, xg, nullptr, 0, G, dc, stream);
}

void launch_sym_contract_sets(int S, int N, int L1, int64_t n_sets, const SymSets& sets, const double* c,
                              const double* norm2, const double* E, const double* T, double* dc,
                              hipStream_t stream) {
  if (n_sets == 0 || sets.n_ids == 0) return;
  if (n_sets > 65535) throw InvalidArgument("too many sets in one launch");
  const int R = S * N;
  const size_t smem = sizeof(double) * size_t(sym_tri(R));
  auto go = [&](auto kern, size_t smem) {
    allow_lds(kern, smem);
    // (channels over more workgroups where there are few: 4 points of 42 centres in 4
    // species, n_max 9, l_max 9, whole call 0.98 -> 0.42 ms)
    const int64_t blocks = (sets.n_ids + kSetCentres - 1) / kSetCentres * n_sets;
    const unsigned split = unsigned(std::max<int64_t>(1, std::min<int64_t>(L1, 512 / blocks)));
    hipLaunchKernelGGL(kern, dim3(unsigned((sets.n_ids + kSetCentres - 1) / kSetCentres), unsigned(n_sets), split),
                       dim3(kThreads), smem, stream, R, N, L1 - 1, sym_row_stride(S, N, L1), sets, c, norm2, E, T, dc);
    RGPU_LAUNCH_CHECK();
  };
  if (smem <= kContractLds)
    go(sym_contract_sets_kernel<true>, smem);
  else
    go(sym_contract_sets_kernel<false>, 0);
}

void launch_sym_contract_full(int S, int N, int L1, int64_t n, const double* c, const double* p, const double* norm2,
                              const double* G, DeviceBuffer<double>& work, double* dc, hipStream_t stream) {
  if (n == 0) return;
  const int R = S * N;
  const size_t whole = sizeof(double) * size_t(L1) * full_stride(R) + sizeof(int) * size_t(S) * (S + 1) / 2;
  if (whole <= kFullLds) {
    auto go = [&](auto kern) {
      allow_lds(kern, whole);
      hipLaunchKernelGGL(kern, dim3(unsigned(n)), dim3(kThreads), whole, stream, R, N, L1 - 1,
                         sym_row_stride(S, N, L1), c, p, norm2, G, dc);
      RGPU_LAUNCH_CHECK();
    };
    if (L1 <= 10)
      go(sym_contract_full_kernel<9>);
    else
      go(sym_contract_full_kernel<kMaxL1 - 1>);
    return;
  }
  // Packed first, with p . G where that is needed.  (A form that took the full
  // row's entries channel by channel, L+1 values apart, touched every cache line
  // L+1 times.)
  const int64_t ld = sym_row_stride(S, N, L1);
  const unsigned split = row_split(S, N, L1, n);
  double* g = work.reserve(size_t(n * ld + n * split));
  if (p) {
    go_pack<kDot>(S, N, L1, n, split, G, nullptr, g, nullptr, p, g + n * ld, stream);
    go_contract<true>(S, N, L1, n, c, p, norm2, nullptr, g + n * ld, int(split), g, dc, stream);
  } else {
    go_pack<kPlain>(S, N, L1, n, split, G, nullptr, g, nullptr, nullptr, nullptr, stream);
    go_contract<false>(S, N, L1, n, c, nullptr, nullptr, nullptr, nullptr, 0, g, dc, stream);
  }
}

void launch_sym_pack(int S, int N, int L1, int64_t n, const double* full, const int64_t* rows, double* out,
                     hipStream_t stream, int* asymmetric) {
  if (n == 0) return;
  const unsigned split = row_split(S, N, L1, n);
  if (asymmetric)
    go_pack<kCheck>(S, N, L1, n, split, full, rows, out, asymmetric, nullptr, nullptr, stream);
  else
    go_pack<kPlain>(S, N, L1, n, split, full, rows, out, nullptr, nullptr, nullptr, stream);
}

void launch_sym_unpack(int S, int N, int L1, int64_t n, const double* p, const int64_t* rows, const double* norm2,
                       bool normalize, double* out, hipStream_t stream) {
  if (n == 0) return;
  const size_t smem = key_lds(S, N, L1);
  allow_lds(sym_unpack_kernel, smem);
  hipLaunchKernelGGL(sym_unpack_kernel, dim3(unsigned(n), row_split(S, N, L1, n)), dim3(kThreads), smem, stream, S, N, L1,
                     key_blocks(S, N, L1), sym_row_stride(S, N, L1), p, rows, norm2, int(normalize), out);
  RGPU_LAUNCH_CHECK();
}

}  // namespace rgpu
