// Pair phase of the adjoint, and the expansion, by wavefronts
// (pair_kernels.hh).
//
// Lanes stand for the (l, mu) of the spherical harmonics, mu = 0 .. l: a lane
// holds dL/dc of its two orders +-mu for every radial channel of one
// neighbour species in registers, so a pair costs it 4 FMAs per channel with
// operands {R, W} that all lanes of one l share (16-byte LDS reads), and no
// other traffic.  The layout this replaced gave a lane one radial channel and
// read dL/dc and the harmonics of every order from LDS, 20 bytes for 4 FMAs,
// which bounded it; the chain from staging a batch to its sums does now, with
// 3 (FP64) or 4 wavefronts per SIMD.  Before and after: FP32, n_max 12,
// l_max 9, 8192 centres of 27 neighbours 282 and 174 us (204 with 31 neighbours);
// FP64, 4096 centres 332 and 162 us, n_max 10, l_max 8, 1024 centres 61 and 52
// us, 64 centres of n_max 8, l_max 6 24 and 17 us.
//
// A wavefront takes its centre's pairs 64 at a time, a lane each for the pair
// records and the final force, and works through them species by species in
// batches of four: their harmonics (one lane per pair and order m >= 0) and
// radial functions (all lanes over the (n, l) of one pair, whose spline cell
// and weights are then wavefront-uniform) are formed in LDS, then contracted.
// With (l_max+1)(l_max+2)/2 <= 32 or 16 units, two or four pairs are
// contracted side by side.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "pair_kernels.hh"
#include "soap_device.hh"

namespace rgpu {

namespace {

constexpr int kThreads = 256, kWaves = kThreads / 64;
constexpr int kBatch = 4;     // pairs staged at a time
constexpr int kMaxPairL = 9;  // (l, mu) units fit a wavefront

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int lane_value(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  const int2 b = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(b.x, lane),
                                              __builtin_amdgcn_readlane(b.y, lane)));
}

// recursion coefficients of Y_lm (radial.hh), and the gradient terms
template <class T>
__device__ __forceinline__ const T* ylm_src(const RadialDev& R);
template <>
__device__ __forceinline__ const double* ylm_src<double>(const RadialDev& R) { return R.ylm64; }
template <>
__device__ __forceinline__ const float* ylm_src<float>(const RadialDev& R) { return R.ylm32; }
template <class T>
__device__ __forceinline__ const YGradTerm<T>* ygrad_of(const RadialDev& R);
template <>
__device__ __forceinline__ const YGradTerm<double>* ygrad_of<double>(const RadialDev& R) { return R.ygrad64; }
template <>
__device__ __forceinline__ const YGradTerm<float>* ygrad_of<float>(const RadialDev& R) { return R.ygrad32; }

template <class T>
struct Vec2;
template <>
struct Vec2<float> {
  typedef float type __attribute__((ext_vector_type(4)));  // {R, W} of two channels
};
template <>
struct Vec2<double> {
  typedef double type __attribute__((ext_vector_type(2)));  // {R, W} of one channel
};

// One pair's record, a lane each: direction, species, spline cell, and what
// turns the cell's {y0, d0, y1, d1} into R fc / r = ra y0 + rb d0 + rc y1 +
// rd d1 and W = R' fc + R fc' = we (y1 - y0) + wa y0 + wb d0 + wc y1 + wd d1
// (math/interpolator.hh:166-186; the difference is formed first: its factor
// is the inverse grid spacing).
template <class T>
struct PairRec {
  T x, y, z;
  T ra, rb, rc, rd, we, wa, wb, wc, wd;
  int sp, klo;
};

template <class T>
__device__ __forceinline__ PairRec<T> load_pair(const RadialDev& rad, const PairView& pv, int64_t p) {
  PairRec<T> r;
  const double d = pv.pair_dist[p], fc = pv.pair_fc[p], dfc = pv.pair_dfc[p];
  r.sp = pv.species_of[pv.pair_j[p]];
  r.x = T(pv.pair_vec[3 * p] / d);
  r.y = T(pv.pair_vec[3 * p + 1] / d);
  r.z = T(pv.pair_vec[3 * p + 2] / d);
  double xhi, h;
  r.klo = spline_cell_of(rad, d, r.sp, &xhi, &h);
  const double a = (xhi - d) / h, b = 1 - a, fr = fc / d, fh = fc / h;
  const double ca = a * (a * a - 1), cb = b * (b * b - 1);
  r.ra = T(a * fr);
  r.rb = T(ca * fr);
  r.rc = T(b * fr);
  r.rd = T(cb * fr);
  r.we = T(fh);
  r.wa = T(a * dfc);
  r.wb = T(ca * dfc - (3 * a * a - 1) * fh);
  r.wc = T(b * dfc);
  r.wd = T(cb * dfc + (3 * b * b - 1) * fh);
  return r;
}

// the same for the expansion: R fc = ra y0 + rb d0 + rc y1 + rd d1
template <class T>
struct PairValue {
  T x, y, z;
  T ra, rb, rc, rd;
  int sp, klo;
};

template <class T>
__device__ __forceinline__ PairValue<T> load_pair_value(const RadialDev& rad, const PairView& pv, int64_t p) {
  PairValue<T> r;
  const double d = pv.pair_dist[p], fc = pv.pair_fc[p];
  r.sp = pv.species_of[pv.pair_j[p]];
  r.x = T(pv.pair_vec[3 * p] / d);
  r.y = T(pv.pair_vec[3 * p + 1] / d);
  r.z = T(pv.pair_vec[3 * p + 2] / d);
  double xhi, h;
  r.klo = spline_cell_of(rad, d, r.sp, &xhi, &h);
  const double a = (xhi - d) / h, b = 1 - a;
  r.ra = T(a * fc);
  r.rb = T(a * (a * a - 1) * fc);
  r.rc = T(b * fc);
  r.rd = T(b * (b * b - 1) * fc);
  return r;
}

// the next kBatch pairs of a mask (their lanes), and how many there are
__device__ __forceinline__ int next_batch(unsigned long long& mask, int (&q)[kBatch]) {
  int nb = 0;
#pragma unroll
  for (int b = 0; b < kBatch; ++b) {
    q[b] = mask ? __ffsll((long long)mask) - 1 : 0;
    nb += mask ? 1 : 0;
    mask &= mask - 1;
  }
  return nb;
}

// Recursion table of the harmonics in LDS, [L1][L1] x {a, a b, start, 0}:
// with Q_m(l) = P_lm / sin^m, Q(l) = a z Q(l-1) + a b Q(l-2) + start, all zero
// below l = m and start the product of the diagonal factors at l = m
// (spherical_harmonics.cc:36-96, the factors sin^m and e^{i m phi} taken out).
template <class T>
__device__ __forceinline__ void fill_ylm_table(const RadialDev& rad, T* dst) {
  const int L1 = rad.L1;
  const T* src = ylm_src<T>(rad);  // ylm_coefficients()
  const T *dfac = src + 4 * L1 * L1, *s2l1 = dfac + L1;
  for (int e = threadIdx.x; e < L1 * L1; e += blockDim.x) {
    const int l = e / L1, m = e - l * L1;
    T a = T(0), ab = T(0), st = T(0);
    if (m == l) {
      st = T(0.39894228040143267794);
      for (int k = 1; k <= m; ++k) st *= dfac[k];
    } else if (m == l - 1) {
      a = s2l1[l];
    } else if (m < l - 1) {
      a = src[4 * e];
      ab = a * src[4 * e + 1];
    }
    dst[4 * e] = a;
    dst[4 * e + 1] = ab;
    dst[4 * e + 2] = m == 0 ? st * T(0.70710678118654752440) : st;  // m = 0: 1 / sqrt 2
    dst[4 * e + 3] = T(0);
  }
}

// Y_l^{+-m}, l = m .. L, of a unit direction on the lane of order m (<= 15),
// written to Y[l*l + l +- m]: Q_m(l) times the real and imaginary part of
// (x + i y)^m
template <class T>
__device__ __forceinline__ void ylm_of_order(int L, const T* __restrict__ tab, T x, T y, T z, int m, bool on, T* Y) {
  typedef T V4 __attribute__((ext_vector_type(4)));
  const int L1 = L + 1;
  T c = T(1), s = T(0), px = x, py = y;
#pragma unroll
  for (int bit = 1; bit <= 8; bit *= 2) {
    const T cn = c * px - s * py, sn = c * py + s * px;
    const bool use = (m & bit) != 0;
    c = use ? cn : c;
    s = use ? sn : s;
    if (bit < 8) {
      const T q = px * px - py * py;
      py = T(2) * px * py;
      px = q;
    }
  }
  const int mm = m < L1 ? m : 0;
  T P1 = T(0), P2 = T(0);
  for (int l = 0; l <= L; ++l) {
    const V4 q = reinterpret_cast<const V4*>(tab)[l * L1 + mm];
    const T P = (q.x * z) * P1 + (q.y * P2 + q.z);
    if (on && m <= l) {
      const int base = l * l + l;
      Y[base + m] = P * c;
      if (m) Y[base - m] = P * s;
    }
    P2 = P1;
    P1 = P;
  }
}

// --- sums over the lanes -------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  const int b = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const int2 b = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(b.x, b.x, CTRL, 0xf, 0xf, false),
                                              __builtin_amdgcn_update_dpp(b.y, b.y, CTRL, 0xf, 0xf, false)));
}
// quad_perm xor 1 and xor 2; mirrors in 8 and 16 lanes (xor 4 and xor 8 once
// the smaller groups hold equal values); rotation by 8 in 16 lanes (xor 8)
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kHalfMirror = 0x141, kMirror = 0x140, kRor8 = 0x128;

// a + b halved over the lanes: the lanes with bit 32 (16) clear get a summed
// over that bit, the others b
template <int BIT>
__device__ __forceinline__ unsigned swap_half(unsigned& a, unsigned b) {
  if constexpr (BIT == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    return r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    return r[1];
  }
}
template <int BIT>
__device__ __forceinline__ float halve(float a, float b) {
  unsigned x = __builtin_bit_cast(unsigned, a);
  const unsigned y = swap_half<BIT>(x, __builtin_bit_cast(unsigned, b));
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
template <int BIT>
__device__ __forceinline__ double halve(double a, double b) {
  uint2 x = __builtin_bit_cast(uint2, a);
  const uint2 v = __builtin_bit_cast(uint2, b);
  const uint2 y = make_uint2(swap_half<BIT>(x.x, v.x), swap_half<BIT>(x.y, v.y));
  return __builtin_bit_cast(double, x) + __builtin_bit_cast(double, y);
}

// Sums v0 .. v3 over aligned groups of G lanes: on return the k-th quarter of
// a group holds the sum of v_k (quarters in the order of the two lane bits
// that were halved first, G 16: bits 8 and 4).
template <int G, class T>
__device__ __forceinline__ T group_sums(T v0, T v1, T v2, T v3, int lane) {
  if constexpr (G == 64) {
    T t = halve<16>(halve<32>(v0, v2), halve<32>(v1, v3));
    t += dpp<kXor1>(t);
    t += dpp<kXor2>(t);
    t += dpp<kHalfMirror>(t);
    return t + dpp<kMirror>(t);
  } else if constexpr (G == 32) {
    const T a = halve<16>(v0, v2), b = halve<16>(v1, v3);
    const bool q = (lane & 8) != 0;
    T t = (q ? b : a) + dpp<kRor8>(q ? a : b);
    t += dpp<kXor1>(t);
    t += dpp<kXor2>(t);
    return t + dpp<kHalfMirror>(t);
  } else {
    T v[4] = {v0, v1, v2, v3};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] += dpp<kXor1>(v[k]);
      v[k] += dpp<kXor2>(v[k]);
    }
    const bool h = (lane & 8) != 0, q = (lane & 4) != 0;
    const T a = (h ? v[2] : v[0]) + dpp<kRor8>(h ? v[0] : v[2]);
    const T b = (h ? v[3] : v[1]) + dpp<kRor8>(h ? v[1] : v[3]);
    return (q ? b : a) + dpp<kHalfMirror>(q ? a : b);
  }
}

// Wavefronts per SIMD that the registers are shared out for.  Past 16 channels
// (FP64: past 12) a lane's channels spilled at the usual number (24 channels
// in FP64: 80 to 105 registers): 4520 centres of 3 species, n_max 20, l_max 2,
// FP64 expansion with the features 199 -> 156 us; the adjoint of 700 centres,
// n_max 24, l_max 2, 109 -> 95 us.
template <class T, int NT>
__host__ __device__ constexpr int force_waves() {
  return sizeof(T) == 4 ? (NT <= 16 ? 4 : 3) : (NT <= 12 ? 3 : 2);
}
template <class T, int NT>
__host__ __device__ constexpr int expansion_waves() {
  return sizeof(T) == 4 ? (NT <= 16 ? 5 : 4) : (NT <= 12 ? 4 : (NT <= 16 ? 3 : 2));
}

// per-wavefront LDS of the pair phase
template <class T, int NT>
__host__ __device__ inline size_t force_wave_lds(int L1) {
  return sizeof(T) * (size_t(kBatch) * (((L1 * L1) + 1) / 2 * 2 + size_t(L1) * 2 * NT) + 4 * 64);
}

// NT: radial channels rounded up (the surplus ones zero); G: lanes per pair;
// W: wavefronts per centre
template <class T, int NT, int G, int W>
__global__ __launch_bounds__(kThreads, (force_waves<T, NT>())) void pair_force_kernel(RadialDev rad, int S, PairView pv,
                                                              const T* __restrict__ dcg,
                                                              double* __restrict__ centre_virial) {
  typedef typename Vec2<T>::type V;
  typedef T V4 __attribute__((ext_vector_type(4)));
  constexpr int PPI = 64 / G;  // pairs side by side
  const int N = rad.N, L = rad.L, L1 = rad.L1, LL = rad.LL, F = N * L1, LP = (LL + 1) / 2 * 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  extern __shared__ __align__(64) unsigned char smem_raw[];
  T* yc = reinterpret_cast<T*>(smem_raw);
  T* Y = yc + 4 * LL + wave * (force_wave_lds<T, NT>(L1) / sizeof(T));
  T* RW = Y + kBatch * LP;            // [batch][l][NT]{R fc / r, R' fc + R fc'}
  T* res = RW + kBatch * L1 * 2 * NT;  // [64][4]
  __shared__ double red[kWaves][9];  // centre force and virial of each wavefront
  fill_ylm_table<T>(rad, yc);
  for (int e = lane; e < kBatch * L1 * 2 * NT; e += 64) RW[e] = T(0);  // surplus channels stay zero
  if (lane < 9) red[wave][lane] = 0.0;
  __syncthreads();

  // this lane's unit (l, mu) and its orders +mu, -mu (mu 0: one order)
  const int un = lane & (G - 1), grp = lane / G;
  int l = 0;
  while ((l + 1) * (l + 2) / 2 <= un) ++l;
  const bool unit = l <= L;
  if (!unit) l = 0;
  const int mu = unit ? un - l * (l + 1) / 2 : 0;
  const int lp = l * l + l + mu, lm = l * l + l - mu;
  // harmonics of degree l - 1 and orders mu - 1, mu, mu + 1 (cos and sin) that
  // the gradients of this lane's two are made of, and their coefficients
  const int b1 = (l - 1) * l;
  auto at = [&](int m, bool ok) { return ok && l > 0 ? b1 + m : 0; };
  const int ic0 = at(mu - 1, mu >= 1), ic1 = at(mu, mu <= l - 1), ic2 = at(mu + 1, mu + 1 <= l - 1);
  const int is0 = at(-(mu - 1), mu >= 2), is1 = at(-mu, mu >= 1 && mu <= l - 1), is2 = at(-(mu + 1), mu + 1 <= l - 1);
  const YGradTerm<T>* gt = ygrad_of<T>(rad);
  auto coef = [&](int q, int c, int idx, bool ok) -> T {
    if (!unit || !ok || l == 0) return T(0);
    const YGradTerm<T> g = gt[3 * q + c];
    return (g.c0 != T(0) && g.i0 == idx ? g.c0 : T(0)) + (g.c1 != T(0) && g.i1 == idx ? g.c1 : T(0));
  };
  const bool k0 = mu >= 1, k2 = mu + 1 <= l - 1, z0 = mu >= 2;
  const T px0 = coef(lp, 0, ic0, k0), px2 = coef(lp, 0, ic2, k2);
  const T py0 = coef(lp, 1, is0, z0), py2 = coef(lp, 1, is2, k2);
  const T pz1 = coef(lp, 2, ic1, mu <= l - 1);
  const T mx0 = mu ? coef(lm, 0, is0, z0) : T(0), mx2 = mu ? coef(lm, 0, is2, k2) : T(0);
  const T my0 = mu ? coef(lm, 1, ic0, k0) : T(0), my2 = mu ? coef(lm, 1, ic2, k2) : T(0);
  const T mz1 = mu ? coef(lm, 2, is1, mu <= l - 1) : T(0);
  const T tl = T(l);
  const float inv_n = 1.0f / float(N);
  const int seg = lane / L1, mo = lane - seg * L1;  // staging: pair and order of the harmonics

  // a wavefront takes several centres in turn (W > 1: its workgroup's one)
  constexpr int per = kWaves / W;
  const int w = W > 1 ? wave % W : 0;
  for (int64_t i0 = int64_t(blockIdx.x) * per; i0 < pv.n_centres; i0 += int64_t(gridDim.x) * per) {
    const int64_t v = i0 + wave / W;
    if (W == 1 && v >= pv.n_centres) break;
    const bool live = v < pv.n_centres;  // (W > 1: every wavefront reaches the barriers)
    const PairEntry entry = pair_entry(pv, live ? v : pv.n_centres - 1);
    const int64_t i = entry.centre;
    const int64_t p0 = pv.centre_off[i] + 1;  // the self pair contributes nothing
    const int np = live ? int(pv.centre_off[i + 1] - p0) : 0;
    const T* dci = dcg + v * int64_t(S) * LL * N;
    const V4* table = Spl4<T>::table(rad);
    for (int c0 = 0; c0 < np; c0 += 64 * W) {
      const int k = c0 + lane * W + w;
      const bool act = k < np;
      const int64_t p = p0 + (act ? k : 0);
      const PairRec<T> rec = load_pair<T>(rad, pv, p);
      unsigned long long todo = __ballot(act);
      while (todo) {
        // the pairs of one neighbour species
        const int s = lane_value(rec.sp, __ffsll((long long)todo) - 1);
        unsigned long long mine = __ballot(act && rec.sp == s) & todo;
        todo &= ~mine;
        T cp[NT], cm[NT];
        {
          // (rows read NT values: the surplus ones lie in the next row, the
          // last row's in the buffer's slack, and are dropped)
          const T* r = dci + int64_t(s) * LL * N;
          const T *rp = r + lp * N, *rm = r + lm * N;
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            const T vp = rp[n], vm = rm[n];
            cp[n] = unit && n < N ? vp : T(0);
            cm[n] = unit && mu && n < N ? vm : T(0);
          }
        }
        while (mine) {
          int q[kBatch];
          const int nb = next_batch(mine, q);
          wave_sync();  // the previous batch is read
          {
            const int src = seg == 0 ? q[0] : (seg == 1 ? q[1] : (seg == 2 ? q[2] : q[3]));
            const T x = __shfl(rec.x, src, 64), y = __shfl(rec.y, src, 64), z = __shfl(rec.z, src, 64);
            ylm_of_order<T>(L, yc, x, y, z, mo, seg < nb, Y + seg * LP);
          }
          for (int e = lane; e < F; e += 64) {
            const int el = int((float(e) + 0.5f) * inv_n), en = e - el * N;
            V4 t[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; ++b)
              t[b] = table[int64_t(lane_value(rec.klo, q[b])) * F + en * L1 + el];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
              if (b >= nb) continue;
              const V4 y = t[b];
              const int k = q[b];
              T r = lane_value(rec.ra, k) * y.x, v = lane_value(rec.wa, k) * y.x;
              r += lane_value(rec.rb, k) * y.y;
              v += lane_value(rec.wb, k) * y.y;
              r += lane_value(rec.rc, k) * y.z;
              v += lane_value(rec.wc, k) * y.z;
              r += lane_value(rec.rd, k) * y.w;
              v += lane_value(rec.wd, k) * y.w;
              v += lane_value(rec.we, k) * (y.z - y.x);
              T* o = RW + ((b * L1 + el) * NT + en) * 2;
              o[0] = r;
              o[1] = v;
            }
          }
          wave_sync();
#pragma unroll 1
          for (int b0 = 0; b0 < nb; b0 += PPI) {
            const int b = b0 + grp;
            const T* Yb = Y + b * LP;
            const V* rw = reinterpret_cast<const V*>(RW + (b * L1 + l) * 2 * NT);
            T Vp = T(0), Vm = T(0), Wp = T(0), Wm = T(0);
            if constexpr (sizeof(T) == 4) {
#pragma unroll
              for (int n = 0; n < NT; n += 2) {
                const V x = rw[n / 2];
                Vp += cp[n] * x.x;
                Wp += cp[n] * x.y;
                Vm += cm[n] * x.x;
                Wm += cm[n] * x.y;
                Vp += cp[n + 1] * x.z;
                Wp += cp[n + 1] * x.w;
                Vm += cm[n + 1] * x.z;
                Wm += cm[n + 1] * x.w;
              }
            } else {
#pragma unroll
              for (int n = 0; n < NT; ++n) {
                const V x = rw[n];
                Vp += cp[n] * x.x;
                Wp += cp[n] * x.y;
                Vm += cm[n] * x.x;
                Wm += cm[n] * x.y;
              }
            }
            const T yp = Yb[lp], ym = Yb[lm];
            const T yc0 = Yb[ic0], yc1 = Yb[ic1], yc2 = Yb[ic2], ys0 = Yb[is0], ys1 = Yb[is1], ys2 = Yb[is2];
            // A - Sl = sum (W - l V) Y, B_c = sum V gY_c (a slot without a pair
            // holds stale values; its sums are not kept)
            const T t = group_sums<G>((Wp - tl * Vp) * yp + (Wm - tl * Vm) * ym,
                                      Vp * (px0 * yc0 + px2 * yc2) + Vm * (mx0 * ys0 + mx2 * ys2),
                                      Vp * (py0 * ys0 + py2 * ys2) + Vm * (my0 * yc0 + my2 * yc2),
                                      Vp * (pz1 * yc1) + Vm * (mz1 * ys1), lane);
            const int dst = b == 0 ? q[0] : (b == 1 ? q[1] : (b == 2 ? q[2] : q[3]));
            if ((lane & (G / 4 - 1)) == 0 && b < nb) res[4 * dst + (lane & (G - 1)) / (G / 4)] = t;
          }
        }
      }
      wave_sync();  // every pair's sums in place
      double r[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
      if (act) {
        const double vx = pv.pair_vec[3 * p], vy = pv.pair_vec[3 * p + 1], vz = pv.pair_vec[3 * p + 2];
        const double Q = double(res[4 * lane]) / pv.pair_dist[p];
        const double g[3] = {Q * vx + double(res[4 * lane + 1]), Q * vy + double(res[4 * lane + 2]),
                             Q * vz + double(res[4 * lane + 3])};
        double* pf = pv.pair_force + 3 * (entry.set * pv.set_pairs + p);
        pf[0] = g[0];
        pf[1] = g[1];
        pf[2] = g[2];
        if (pv.pair_j[p] != int(i)) {
          r[0] = -g[0];
          r[1] = -g[1];
          r[2] = -g[2];
        }
        // r_ji = r_i - r_j(image) = -pair vector
        r[3] = -vx * g[0];
        r[4] = -vy * g[1];
        r[5] = -vz * g[2];
        r[6] = -vy * g[2];
        r[7] = -vz * g[0];
        r[8] = -vx * g[1];
      }
      // (per chunk, in a fixed order: nothing of this lives across the batches)
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        for (int off = 32; off > 0; off >>= 1) r[k] += __shfl_xor(r[k], off, 64);
        if (lane == 0) red[wave][k] += r[k];
      }
      wave_sync();  // res is read before the next chunk writes it
    }
    if constexpr (W > 1)
      __syncthreads();
    else
      wave_sync();
    if (w == 0 && live && lane < 9) {
      double t = 0;
#pragma unroll
      for (int k = 0; k < W; ++k) t += red[wave + k][lane];
      const int64_t o = entry.set * pv.set_centres + i;
      if (lane < 3)
        pv.centre_force[3 * o + lane] = t;
      else
        centre_virial[6 * o + lane - 3] = t;
    }
    if constexpr (W > 1) __syncthreads();
    if (lane < 9) red[wave][lane] = 0.0;
    wave_sync();
  }
}

// Row stride of the expansion's radial functions in LDS: whole vectors, so that
// every row is aligned for the vector reads and the last one's end inside.
template <class T, int NT>
__host__ __device__ constexpr int expansion_row() {
  constexpr int VN = sizeof(typename Vec2<T>::type) / sizeof(T);
  return (NT + VN - 1) / VN * VN;
}

// Expansion c[i][s][n][lm] = [s == s_i][lm == 0] R0[n] / sqrt(4 pi) + sum over
// the pairs (i, j), s_j = s, of fc R_nl Y_lm, with the layout of the pair
// phase: a lane holds the sums of its two orders +-mu for every radial channel
// in registers, two FMAs per channel and pair whose radial operand all lanes
// of one l share.  (The per-entry kernel reads both operands of every FMA from
// LDS, which bounds it; the staging of a batch bounds this one.)  One
// wavefront per centre, several in turn: 178 -> 93 us for 8192 centres
// of 27 neighbours, n_max 12, l_max 9, FP32 (104 with 31); 167 -> 72 us for 4096
// centres, FP64.
template <class T, int NT>
__host__ __device__ inline size_t expansion_wave_lds(int L1) {
  return sizeof(T) * (size_t(kBatch) * (((L1 * L1) + 1) / 2 * 2 + size_t(L1) * expansion_row<T, NT>()));
}

template <class T, int NT, int G>
__global__ __launch_bounds__(kThreads, (expansion_waves<T, NT>())) void expansion_wave_kernel(
    RadialDev rad, int S, PairView pv, T* __restrict__ cout, unsigned long long* __restrict__ keymask) {
  typedef typename Vec2<T>::type V;
  typedef T V4 __attribute__((ext_vector_type(4)));
  constexpr int PPI = 64 / G, VN = sizeof(V) / sizeof(T), NR = expansion_row<T, NT>();
  static_assert(NR % VN == 0 && NR >= NT, "rows are read as vectors");
  const int N = rad.N, L = rad.L, L1 = rad.L1, LL = rad.LL, F = N * L1, LP = (LL + 1) / 2 * 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  extern __shared__ __align__(64) unsigned char smem_raw[];
  T* yc = reinterpret_cast<T*>(smem_raw);
  T* Y = yc + 4 * LL + wave * (expansion_wave_lds<T, NT>(L1) / sizeof(T));
  T* R = Y + kBatch * LP;  // [batch][l][NR]
  fill_ylm_table<T>(rad, yc);
  for (int e = lane; e < kBatch * L1 * NR; e += 64) R[e] = T(0);  // surplus channels stay zero
  __syncthreads();
  const int un = lane & (G - 1), grp = lane / G;
  int l = 0;
  while ((l + 1) * (l + 2) / 2 <= un) ++l;
  const bool unit = l <= L;
  if (!unit) l = 0;
  const int mu = unit ? un - l * (l + 1) / 2 : 0;
  const int lp = l * l + l + mu, lm = l * l + l - mu;
  const int seg = lane / L1, mo = lane - seg * L1;
  const float inv_n = 1.0f / float(N);
  const V4* table = Spl4<T>::table(rad);
  const double inv_s4pi = 0.28209479177387814347;  // 1/sqrt(4 pi)

  for (int64_t i = int64_t(blockIdx.x) * kWaves + wave; i < pv.n_centres; i += int64_t(gridDim.x) * kWaves) {
    const int64_t p0 = pv.centre_off[i] + 1;  // the self pair contributes nothing here
    const int np = int(pv.centre_off[i + 1] - p0);
    const int si = pv.species_of[i];
    T* ci = cout + i * int64_t(S) * N * LL;
    unsigned long long present = 1ull << si;
    for (int c0 = 0; c0 == 0 || c0 < np; c0 += 64) {
      const bool act = c0 + lane < np;
      PairValue<T> rec{};
      rec.sp = -1;
      if (act) rec = load_pair_value<T>(rad, pv, p0 + c0 + lane);
      for (int s = 0; s < S; ++s) {
        unsigned long long mine = __ballot(rec.sp == s);
        if (c0 > 0 && !mine) continue;
        if (mine) present |= 1ull << s;
        T ap[NT], am[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) ap[n] = am[n] = T(0);
        while (mine) {
          int q[kBatch];
          const int nb = next_batch(mine, q);
          wave_sync();  // the previous batch is read
          {
            const int src = seg == 0 ? q[0] : (seg == 1 ? q[1] : (seg == 2 ? q[2] : q[3]));
            const T x = __shfl(rec.x, src, 64), y = __shfl(rec.y, src, 64), z = __shfl(rec.z, src, 64);
            ylm_of_order<T>(L, yc, x, y, z, mo, seg < nb, Y + seg * LP);
          }
          for (int e = lane; e < F; e += 64) {
            const int el = int((float(e) + 0.5f) * inv_n), en = e - el * N;
            V4 t[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; ++b)
              t[b] = table[int64_t(lane_value(rec.klo, q[b])) * F + en * L1 + el];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
              T r = lane_value(rec.ra, q[b]) * t[b].x;
              r += lane_value(rec.rb, q[b]) * t[b].y;
              r += lane_value(rec.rc, q[b]) * t[b].z;
              r += lane_value(rec.rd, q[b]) * t[b].w;
              R[(b * L1 + el) * NR + en] = b < nb ? r : T(0);
            }
          }
          wave_sync();
          // (an empty slot's radial functions are zero; its harmonics may be
          // stale, of an earlier pair or never written: they are not read)
#pragma unroll 1
          for (int b0 = 0; b0 < nb; b0 += PPI) {
            const int b = b0 + grp;
            const bool on = unit && b < nb;
            const T yp = on ? Y[b * LP + lp] : T(0), ym = on ? Y[b * LP + lm] : T(0);
            const V* r = reinterpret_cast<const V*>(R + (b * L1 + l) * NR);
#pragma unroll
            for (int n = 0; n < NT; n += VN) {
              const V x = r[n / VN];
#pragma unroll
              for (int k = 0; k < VN; ++k) {
                if (n + k < NT) {
                  ap[n + k] += x[k] * yp;
                  am[n + k] += x[k] * ym;
                }
              }
            }
          }
        }
        // the groups' sums; then this species' block
        T* cs = ci + int64_t(s) * N * LL;
        const double* centre = rad.center + (rad.sp_tab ? rad.sp_tab[si] * N : 0);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          if (n >= N) continue;
          T vp = ap[n], vm = am[n];
          if constexpr (G <= 32) {
            vp += __shfl_xor(vp, 32, 64);
            vm += __shfl_xor(vm, 32, 64);
          }
          if constexpr (G <= 16) {
            vp += __shfl_xor(vp, 16, 64);
            vm += __shfl_xor(vm, 16, 64);
          }
          if (unit && grp == 0) {
            T* o = cs + n * LL;
            if (c0 > 0) {
              vp += o[lp];
              vm += o[lm];
            } else if (s == si && lp == 0) {
              vp += T(centre[n] * inv_s4pi);
            }
            o[lp] = vp;
            if (mu) o[lm] = vm;
          }
        }
      }
    }
    if (lane == 0) keymask[i] = present;
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

// f(std::integral_constant<int, NT>) for the smallest built NT >= N
template <class F>
void with_channels(int N, F&& f) {
  if (N <= 4)
    f(std::integral_constant<int, 4>{});
  else if (N <= 6)
    f(std::integral_constant<int, 6>{});
  else if (N <= 8)
    f(std::integral_constant<int, 8>{});
  else if (N <= 10)
    f(std::integral_constant<int, 10>{});
  else if (N <= 12)
    f(std::integral_constant<int, 12>{});
  else if (N <= 16)
    f(std::integral_constant<int, 16>{});
  else
    f(std::integral_constant<int, kMaxN>{});
}

}  // namespace

bool pair_kernels_apply(const RadialDev& rad) { return rad.use_spline && rad.L <= kMaxPairL && rad.N <= kMaxN; }

template <class T>
void launch_pair_forces(const RadialDev& rad, int S, const PairView& pv, const T* dc, double* centre_virial,
                        hipStream_t stream) {
  const int64_t n = pv.n_centres;
  if (n == 0) return;
  const int units = rad.L1 * (rad.L1 + 1) / 2;
  // As many wavefronts per centre as keep the chip filled: fewer centres share
  // a centre's pairs, whose serial chain shows (one, two, four wavefronts:
  // 64 centres 31, 23, 18 us; 1024 centres 52, 42, 57; 1331 centres in FP32
  // 47, 38, 51; 4096 centres 167, 220, 319 us).
  const int wide = n < 512 ? 4 : (n < 2048 ? 2 : 1);
  with_channels(rad.N, [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    const size_t smem = sizeof(T) * size_t(4 * rad.LL) + kWaves * force_wave_lds<T, NT>(rad.L1);
    auto go = [&](auto kern, int64_t blocks) {
      allow_lds(kern, smem);
      hipLaunchKernelGGL(kern, dim3(unsigned(blocks)), dim3(kThreads), smem, stream, rad, S, pv, dc, centre_virial);
      RGPU_LAUNCH_CHECK();
    };
    // as many workgroups as are resident (by the registers)
    const int64_t resident = int64_t(device_cu_count()) * force_waves<T, NT>();
    auto by_units = [&](auto w) {
      constexpr int W = decltype(w)::value;
      const int64_t blocks = W > 1 ? (n * W + kWaves - 1) / kWaves : std::min((n + kWaves - 1) / kWaves, resident);
      if (units <= 16)
        go(pair_force_kernel<T, NT, 16, W>, blocks);
      else if (units <= 32)
        go(pair_force_kernel<T, NT, 32, W>, blocks);
      else
        go(pair_force_kernel<T, NT, 64, W>, blocks);
    };
    if (wide == 4)
      by_units(std::integral_constant<int, 4>{});
    else if (wide == 2)
      by_units(std::integral_constant<int, 2>{});
    else
      by_units(std::integral_constant<int, 1>{});
  });
}

template <class T>
void launch_expansion_wave(const RadialDev& rad, int S, const PairView& pv, T* c, unsigned long long* keymask,
                           hipStream_t stream) {
  const int64_t n = pv.n_centres;
  if (n == 0) return;
  const int units = rad.L1 * (rad.L1 + 1) / 2;
  with_channels(rad.N, [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    const size_t smem = sizeof(T) * size_t(4 * rad.LL) + kWaves * expansion_wave_lds<T, NT>(rad.L1);
    const int64_t blocks =
        std::min((n + kWaves - 1) / kWaves, int64_t(device_cu_count()) * expansion_waves<T, NT>());
    auto go = [&](auto kern) {
      allow_lds(kern, smem);
      hipLaunchKernelGGL(kern, dim3(unsigned(blocks)), dim3(kThreads), smem, stream, rad, S, pv, c, keymask);
      RGPU_LAUNCH_CHECK();
    };
    if (units <= 16)
      go(expansion_wave_kernel<T, NT, 16>);
    else if (units <= 32)
      go(expansion_wave_kernel<T, NT, 32>);
    else
      go(expansion_wave_kernel<T, NT, 64>);
  });
}
template void launch_expansion_wave<double>(const RadialDev&, int, const PairView&, double*, unsigned long long*,
                                            hipStream_t);
template void launch_expansion_wave<float>(const RadialDev&, int, const PairView&, float*, unsigned long long*,
                                           hipStream_t);
template void launch_pair_forces<double>(const RadialDev&, int, const PairView&, const double*, double*, hipStream_t);
template void launch_pair_forces<float>(const RadialDev&, int, const PairView&, const float*, double*, hipStream_t);

}  // namespace rgpu
