// Fused sweeps of the Wigner split-operator step, ensemble form.
//
//   xsweep  one team per row p:  FFT_x -> kinetic multiplier (p, lambda) -> iFFT_x / X
//           (Fourier_X_To_Lambda_GPU, expPLambda, Fourier_Lambda_To_X_GPU:
//            GPU_Wigner2D_FFT.py:131-158, 788-793, 1885-1888; expPLambdaKinetic,
//            GPU_Wigner2D_GPitaevskii.py:117-158, 1924-1929)
//   psweep  one team per column x of a tile:  FFT_p -> potential multiplier (theta, x)
//           [* Gross-Pitaevskii phase] -> iFFT_p / P -> [Caldeira-Leggett order-3
//           composite] -> [column sums] -> [next Strang half step]
//           (expPotential GPU_Wigner2D_FFT.py:80-126, 795-801, 1891-1913;
//            expPotential_GrossPitaevskii :479-519; theta_fp + CaldeiraDissipatorOrder3
//            :399-431, 1135-1157; GPU_Wigner2D_GPitaevskii.py:60-86, 466-496, 1911-1970)
//   gpshift (rows theta)  G(theta, x) = Re iFFT_x[ FFT_x(rho) (-2i sin(lambda theta/2)) ]
//           (MakeGrossPitaevskiiTerms, GPU_Wigner2D_FFT.py:1687-1705)
//
// Each sweep reads and writes the state once.  Phase multipliers are evaluated
// and applied in FP64 for both state precisions (an FP32 multiplier would be a
// fixed perturbation of the step operator and its error would grow linearly).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "wh_fft.hpp"
#include "wh_kernels.hpp"
#include "wh_math.hpp"
#include "wh_variants.hpp"

namespace wh {

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ double poly(const double* __restrict__ c, int deg, double x) {
  double r = c[deg];
  for (int n = deg - 1; n >= 0; --n) r = fma(r, x, c[n]);
  return r;
}

// Bopp difference of a polynomial V of degree <= kMaxDeg as an odd polynomial in u:
// V(x - u) - V(x + u) = -2 sum_{k odd} D_k(x) u^k, with the Taylor coefficients
// D_k(x) = V^(k)(x) / k! from a Taylor shift of the coefficients c (evaluated once per
// column; each cell then costs four FMAs).  Scaled by f.
struct BoppOdd {
  double e1, e3, e5, e7;
  __device__ __forceinline__ double operator()(double u) const {
    const double u2 = u * u;
    return u * fma(u2, fma(u2, fma(u2, e7, e5), e3), e1);
  }
};
template <class CP>
__device__ __forceinline__ BoppOdd bopp_odd(CP c, int deg, double x, double f) {
  static_assert(kMaxDeg == 8, "odd Taylor terms u, u^3, u^5, u^7");
  double d[kMaxDeg + 1];  // (every row has kMaxDeg + 1 entries: loaded unconditionally, in one go)
#pragma unroll
  for (int n = 0; n <= kMaxDeg; ++n) d[n] = c[n];
#pragma unroll
  for (int n = 0; n <= kMaxDeg; ++n) d[n] = n <= deg ? d[n] : 0.0;
#pragma unroll
  for (int i = 0; i < kMaxDeg; ++i) {
#pragma unroll
    for (int k = kMaxDeg - 1; k >= i; --k) d[k] = fma(x, d[k + 1], d[k]);
  }
  const double g = -2.0 * f;
  return {g * d[1], g * d[3], g * d[5], g * d[7]};
}

// kernel-side FFT-ordered coordinate index: ((k + n/2) mod n) - n/2
__device__ __forceinline__ int fidx(int k, int n) { return ((k + (n >> 1)) & (n - 1)) - (n >> 1); }

// v * m with an FP64 multiplier m; FP32 states are widened for the product.
__device__ __forceinline__ cplx<double> apply(cplx<double> v, cplx<double> m) { return cmul(v, m); }
__device__ __forceinline__ cplx<float> apply(cplx<float> v, cplx<double> m) {
  const double x = v.x, y = v.y;
  return {float(x * m.x - y * m.y), float(x * m.y + y * m.x)};
}
// r * exp(-i phi)
__device__ __forceinline__ cplx<double> expmi(double r, double phi) {
  double s, c;
  sincos_fp64(phi, &s, &c);
  return {r * c, -r * s};
}

template <typename T>
__device__ __forceinline__ cplx<T> scale_load(cplx<T> v, const double* s) {
  return apply(v, cplx<double>{cmem(s)[0], cmem(s)[1]});
}

template <typename T>
__device__ __forceinline__ cplx<T> mul_i(cplx<T> a, T s) { return {-s * a.y, s * a.x}; }

// state storage S <-> arithmetic T (complex64 states with FP64 arithmetic convert at the
// sweep's load and store; every other combination is the identity)
template <typename T, typename S>
__device__ __forceinline__ cplx<T> to_arith(cplx<S> v) {
  return {T(v.x), T(v.y)};
}

// Largest LDS footprint over the supported sizes for a (block, radix) variant: ROWS*Padded(N) =
// (BLOCK/(N/R)) * (N + N/R + 1) elements, and up to 32 more for col_pad.
template <int BLOCK, int R>
constexpr int lds_elems() {
  int m = 0;
  for (int N = 64; N <= 2048; N *= 2) {
    if (N / R > BLOCK || N < R) continue;
    const int rows = BLOCK / (N / R);
    const int e = rows * (N + N / R + 1);
    m = e > m ? e : m;
  }
  return m + 32;
}

template <int N, int R, int BLOCK>
constexpr bool size_ok() {
  return N >= R * 4 && N / R <= BLOCK && BLOCK / (N / R) <= 64;
}

// The (member << 16) | tile item of this block.  A plan of one member computes it: x tiles in
// block order and the record item last; p tiles with consecutive tiles on one XCD (as the work
// lists are cut on the host).
__device__ __forceinline__ unsigned x_item(const SweepArgs& a) {
  if (a.ntiles <= 0) return cmem(a.work)[blockIdx.x];
  return int(blockIdx.x) < a.ntiles ? blockIdx.x : unsigned(kRecordTile);
}
__device__ __forceinline__ unsigned p_item(const SweepArgs& a) {
  if (a.ntiles <= 0) return cmem(a.work)[blockIdx.x];
  const unsigned q = blockIdx.x, nt = unsigned(a.ntiles);
  return nt % 8 == 0 ? (q % 8) * (nt / 8) + q / 8 : q;
}
__device__ __forceinline__ bool first_member(const SweepArgs& a, CMember& m) { return &m == &member_at(a.members, 0); }

// ------------------------------------------------------------------ observables
// Sum over the 64 lanes of a wave (fixed xor tree: deterministic).
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// v from another lane by a DPP control (row = 16 lanes); lanes of rows outside ROWMASK get 0
template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ double dpp_f64(double v) {
  const unsigned long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(unsigned(b)), CTRL, ROWMASK, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, int(unsigned(b >> 32)), CTRL, ROWMASK, 0xF, false);
  return __longlong_as_double((static_cast<unsigned long long>(unsigned(hi)) << 32) | unsigned(lo));
}
// Sum over aligned groups of G lanes (G = 1, 2, 4 .. 64) by VALU lane moves (no LDS
// traffic, fixed order: deterministic); the last lane of each group holds the sum.
//   quad_perm [1,0,3,2], [2,3,0,1]: quad sums;  row_half_mirror: sums of 8;  row_mirror:
//   sums of 16;  row_bcast15 into rows 1, 3: sums of 32 there;  row_bcast31 into rows 2,
//   3: the sum of 64 in row 3.
template <int G>
__device__ __forceinline__ double group_sum(double v) {
  static_assert(G >= 1 && G <= 64 && (G & (G - 1)) == 0, "group of 1..64 lanes");
  if constexpr (G >= 2) v += dpp_f64<0xB1>(v);
  if constexpr (G >= 4) v += dpp_f64<0x4E>(v);
  if constexpr (G >= 8) v += dpp_f64<0x141>(v);
  if constexpr (G >= 16) v += dpp_f64<0x140>(v);
  if constexpr (G >= 32) v += dpp_f64<0x142, 0xA>(v);
  if constexpr (G >= 64) v += dpp_f64<0x143, 0xC>(v);
  return v;
}

// Observable terms of one column from its sums s = (Re S0, Im S0, sum p W, sum p^2 W,
// sum min(W, 0)): the integrands of <x>, <x^2>, <p>, <p^2>, <xp>, <dV/dx>, <p dV/dx>,
// <x dV/dx>, energy, negative area (the per-step record of GPU_Wigner2D_FFT.py:1856-1876).
struct ColumnHost {
  double x, dv, v0;
};
__device__ __forceinline__ ColumnHost column_host(CMember& m, int col) {
  return {gmem(m.x_host)[col], gmem(m.dv_host)[col], gmem(m.v0_host)[col]};
}
__device__ __forceinline__ void column_terms(CMember& m, ColumnHost h, const double (&s)[kNCol],
                                             double (&o)[12]) {
  const double x = h.x, dv = h.dv, v0 = h.v0;
  o[0] = s[0];
  o[1] = s[1];
  o[2] = x * s[0];
  o[3] = x * x * s[0];
  o[4] = s[2];
  o[5] = s[3];
  o[6] = x * s[2];
  o[7] = dv * s[0];
  o[8] = dv * s[2];
  o[9] = x * dv * s[0];
  o[10] = s[3] * m.inv_2m + v0 * s[0];
  o[11] = s[4];
}

// Record row, pending factor and step counter from the 12 observable sums of a member
// (the normalised state is W / n, n = dXdP sum W; observables Re(dXdP sum W A / n)).
__device__ __forceinline__ void write_record(CMember& m, const double (&r)[12], int renorm, int record,
                                             int step) {
  const double nr = m.dxdp * r[0], ni = m.dxdp * r[1];
  double f = 1.0, sr = 1.0, si = 0.0;
  if (renorm) {
    const double m2 = nr * nr + ni * ni;
    f = nr / m2;
    sr = nr / m2;
    si = -ni / m2;
  }
  gmem(m.scale)[0] = sr;
  gmem(m.scale)[1] = si;
  if (record) {
    const gptr<double> o = gmem(m.obs) + size_t(step - m.obs_base) * kNObs;
    const double d = m.dxdp * f;
    o[kObsX] = d * r[2];
    o[kObsX2] = d * r[3];
    o[kObsP] = d * r[4];
    o[kObsP2] = d * r[5];
    o[kObsXP] = d * r[6];
    o[kObsDV] = d * r[7];
    o[kObsPDV] = d * r[8];
    o[kObsXDV] = d * r[9];
    o[kObsH] = d * r[10];
    o[kObsNeg] = d * r[11];
    o[kObsNorm] = d * r[0];
    o[kObsRawNormRe] = nr;
    o[kObsRawNormIm] = ni;
  }
}

// kTilePart epilogue of a p-sweep tile: csum holds the kNCol sums of each of the tile's
// C columns (LDS, visible to every thread: written before a barrier); lane c < C forms the 12
// observable terms of column c (host values h, loaded at the kernel's start) and the lanes' sum
// goes to m.tilepart[k * X + tile].  Tile 0 of member 0 copies the step index to rec_step.
// (One lane per term, each forming every column's terms with the loads of their host values in
// the loop, kept a 128-column tile row of 16 columns busy for 5300 cycles of its 34600.)
template <int C>
__device__ __forceinline__ void write_tile_partial(const SweepArgs& a, CMember& m, int tile,
                                                   const double* csum, ColumnHost h, int step) {
  static_assert(C <= 64, "one wave");
  const int tid = threadIdx.x;
  if (tid < 64) {
    double s[kNCol], o[12];
    const int c = tid % C;
#pragma unroll
    for (int k = 0; k < kNCol; ++k) s[k] = csum[c * kNCol + k];
    column_terms(m, h, s, o);
#pragma unroll
    for (int k = 0; k < 12; ++k) o[k] = group_sum<C>(o[k]);
    if (tid == C - 1) {
#pragma unroll
      for (int k = 0; k < 12; ++k) gmem(m.tilepart)[size_t(k) * m.X + tile] = o[k];
    }
    if (tid == 0 && tile == 0 && first_member(a, m)) *gmem(a.rec_step) = step;  // the step index this sweep read at its start
  }
}

// kTileScale: the x sweep sums the tile partials of the member's last p sweep (every block in
// the same order, so all blocks derive the same factor) into the pending factor 1 / norm (or 1).
// The loads are issued before the state's and the sum is taken when the first transform is done,
// where the factor is needed; the record row is an item of its own.  With the sum in front of the
// transform and the record in tile 0 every block waited for the partials' latency, the wave sums
// and a block barrier (5400 of the 11200 cycles of a 128^2 x sweep): 9.5 -> 4.9 us at 128^2,
// 16.3 -> 15.9 us at 1024^2.
// red: kTileRedBytes of LDS outside the transform arrays.
constexpr int kTileRedBytes = 16 * 12 * 8;
struct TilePartials {
  double re, im;
};
__device__ __forceinline__ int tile_count(const SweepArgs& a, CMember& m) {
  return m.X * (m.P / a.pt_R) / a.pt_block;  // X over the columns per p-sweep tile
}
template <int BLOCK>
__device__ __forceinline__ TilePartials tile_partials(const SweepArgs& a, CMember& m) {
  const int ntiles = tile_count(a, m);
  TilePartials r{0.0, 0.0};
  for (int i = threadIdx.x; i < ntiles; i += BLOCK) {
    r.re += gmem(m.tilepart)[i];
    r.im += gmem(m.tilepart)[size_t(m.X) + i];
  }
  return r;
}
// Contains __syncthreads().
template <int BLOCK>
__device__ __forceinline__ cplx<double> tile_scale(const SweepArgs& a, CMember& m, TilePartials r, double* red) {
  constexpr int kWaves = BLOCK / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  r.re = group_sum<64>(r.re);
  r.im = group_sum<64>(r.im);
  if (lane == 63) {
    red[wave * 2] = r.re;
    red[wave * 2 + 1] = r.im;
  }
  __syncthreads();
  r = {0.0, 0.0};
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    r.re += red[w * 2];
    r.im += red[w * 2 + 1];
  }
  if (!a.fin_renorm) return {1.0, 0.0};
  const double nr = m.dxdp * r.re, ni = m.dxdp * r.im;
  const double m2 = nr * nr + ni * ni;
  return {nr / m2, -ni / m2};
}

// The record item of a member (one block of a kTileScale launch, beside the row tiles so that no
// row waits for it): all 12 sums, the record row and the factor; that of member 0 advances the
// step index.
// AFTER_P: the iteration's p sweep has run (ODM steps, whose join advances the index): the record
// is that of the index before the last p sweep's.
template <int BLOCK, bool AFTER_P = false>
__device__ __forceinline__ void record_item(const SweepArgs& a, CMember& m, double* red) {
  constexpr int kWaves = BLOCK / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ntiles = tile_count(a, m);
  const int rstep = *cmem(a.rec_step) - (AFTER_P ? 1 : 0);  // issued with the partial loads
  double r[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) r[k] = 0.0;
  for (int i = tid; i < ntiles; i += BLOCK) {
#pragma unroll
    for (int k = 0; k < 12; ++k) r[k] += gmem(m.tilepart)[size_t(k) * m.X + i];
  }
#pragma unroll
  for (int k = 0; k < 12; ++k) r[k] = group_sum<64>(r[k]);
  if (lane == 63) {
#pragma unroll
    for (int k = 0; k < 12; ++k) red[wave * 12 + k] = r[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) t += red[w * 12 + k];
    r[k] = t;
  }
  if (tid == 0) {
    write_record(m, r, a.fin_renorm, a.fin_record, rstep);
    if (!AFTER_P && first_member(a, m)) *gmem(a.step) = rstep + 1;
  }
}

// ------------------------------------------------------------------ x sweep
// Kinetic multiplier of element m (lambda index) in row p, linear form:
// exp(-i a m_s), a = dt*dlambda*(k_c0 + k_c1 p), m_s = t + js*TT with
// js = j (j < R/2) or j - R; computed as E_t * Z^js, E_t = exp(-i a t),
// Z = exp(-i a TT): two sincos per lane instead of R.
template <typename T, int R, int TT>
__device__ __forceinline__ void kinetic_apply(cplx<T> (&v)[R], CMember& m, int t, cplx<double> Et, cplx<double> Z1) {
  cplx<double> Zp[R / 2 + 1];  // Z^0 .. Z^(R/2)
  Zp[0] = {1.0, 0.0};
  Zp[1] = Z1;
#pragma unroll
  for (int k = 2; k <= R / 2; ++k) Zp[k] = cmul(Zp[k / 2], Zp[k - k / 2]);
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = apply(v[j], cmul(Et, j < R / 2 ? Zp[j] : cplx<double>{Zp[R - j].x, -Zp[R - j].y}));
  if (m.lambda_decay) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = apply(v[j], cplx<double>{gmem(m.lambda_decay)[t + j * TT], 0.0});
  }
}
template <typename S, typename T, int N, int R, int BLOCK, bool TP, typename E>
__device__ __forceinline__ void xsweep_body(const SweepArgs& a, CMember& m, int tile,
                                            cplx<E>* lds) {
  constexpr int TT = N / R, ROWS = BLOCK / TT;
  constexpr int LSZ = Padded<N, R>::size;
  const int tid = threadIdx.x, team = tid / TT, t = tid % TT;
  const int row = tile * ROWS + team;
  // uniform member base + 32-bit per-lane byte offset (a state is at most 2048^2 x 16 B);
  // the store recomputes the offset from an opaque copy of the lane index, so that no
  // per-row address stays live (or is spilled) across the transforms
  const gptr<cplx<S>> W = gmem(reinterpret_cast<cplx<S>*>(a.W_dst ? a.W_dst : m.W));
  const gptr<const cplx<S>> src = a.W_src ? gmem(reinterpret_cast<const cplx<S>*>(a.W_src)) : gptr<const cplx<S>>(W);
  const unsigned roff = (unsigned(row) * unsigned(N) + unsigned(t)) * unsigned(sizeof(cplx<S>));
  constexpr unsigned kJ = unsigned(TT * sizeof(cplx<S>));
  const Twiddles<T> tw{reinterpret_cast<const cplx<T>*>(m.twX_hi), reinterpret_cast<const cplx<T>*>(m.twX_lo)};
  LdsRow<E> view{lds + team * LSZ};
  // a row's team inside one wave: wave-local exchanges, twiddles loaded once into registers
  // (the throughput form reads them from the table)
  constexpr bool kWave = TT <= 64;
  using Sync = std::conditional_t<kWave, WaveSync, BlockSync>;

  const bool tiles = (a.flags & kTileScale) != 0;
  TilePartials part{0.0, 0.0};
  cplx<double> g{1.0 / N, 0.0};
  if (tiles) {
    part = tile_partials<BLOCK>(a, m);
  } else if (a.flags & kScaleOnLoad) {
    g = {cmem(m.scale)[0] * (1.0 / N), cmem(m.scale)[1] * (1.0 / N)};
  }
  cplx<T> v[R];
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = to_arith<T>(gload<S>(at_off(src, roff + unsigned(j) * kJ)));
  const auto twsrc = [&]() {
    if constexpr (kWave && !TP) {
      TwRegs<T, N, R> r;
      load_twiddles<T, N, R>(r, t, tw);
      return r;
    } else {
      return TwMem<T>{tw};
    }
  }();
  // the two phase factors of the linear form, evaluated while the loads are in flight
  const double p = m.dp * double(fidx(row, m.P));
  const double sgn = (a.flags & kConj) ? -1.0 : 1.0;  // adjoint: conj(r e^{-i phi}) = r e^{+i phi}
  cplx<double> Et{1.0, 0.0}, Z1{1.0, 0.0};
  if (a.kin_linear) {
    const double ak = sgn * a.dt * m.dlambda * (a.k_c0 + a.k_c1 * p);
    Et = expmi(1.0, ak * double(t));
    Z1 = expmi(1.0, ak * double(TT));
  }
  team_fft<T, N, R, -1, LdsRow<E>, Sync>(v, t, view, twsrc);

  // The pending factor and the 1/N of the inverse transform ride on the kinetic
  // multiplier (the transforms are linear): one complex product per lane instead of 2R.
  if (tiles) {
    const cplx<double> f = tile_scale<BLOCK>(a, m, part, reinterpret_cast<double*>(lds + lds_elems<BLOCK, R>()));
    g = {f.x * (1.0 / N), f.y * (1.0 / N)};
  }
  if (a.kin_linear) {
    Et = cmul(Et, g);
    kinetic_apply<T, R, TT>(v, m, t, Et, Z1);
  } else {
    const double hh = a.hbar_half;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int mm = t + j * TT;
      const double lam = m.dlambda * double(fidx(mm, N));
      const double phi = sgn * a.dt * (poly(a.kcoef, a.kdeg, p + hh * lam) - poly(a.kcoef, a.kdeg, p - hh * lam)) * a.inv_hbar;
      const double r = m.lambda_decay ? gmem(m.lambda_decay)[mm] : 1.0;
      v[j] = apply(v[j], cmul(expmi(r, phi), g));
    }
  }
  team_fft<T, N, R, +1, LdsRow<E>, Sync>(v, t, view, twsrc);
  const int ts = opaque_v(int(threadIdx.x));  // offset recomputed from the lane index
  const unsigned soff = (unsigned(tile * ROWS + ts / TT) * unsigned(N) + unsigned(ts % TT)) * unsigned(sizeof(cplx<S>));
#pragma unroll
  for (int j = 0; j < R; ++j) store_stream(at_off(W, soff + unsigned(j) * kJ), to_arith<S>(v[j]));

  if (a.flags & kColPart) {
    // partial column sums of Re W over this tile's rows (Gross-Pitaevskii density after K)
    __syncthreads();
    double* red = reinterpret_cast<double*>(lds);
#pragma unroll
    for (int j = 0; j < R; ++j) red[team * N + t + j * TT] = double(v[j].x);
    __syncthreads();
    for (int x = tid; x < N; x += BLOCK) {
      double s = 0.0;
      for (int q = 0; q < ROWS; ++q) s += red[q * N + x];
      gmem(m.colpart)[size_t(tile) * N + x] = s;
    }
  }
}

// ------------------------------------------------------------------ p sweep
template <typename T, int N, int R, int BLOCK, typename E = T>
struct PSweep {
  static constexpr int TT = N / R;
  static constexpr int C = BLOCK / TT;  // columns per tile
  // wave teams: a column's team lies inside one wave and the transform has an exchange
  // at which the lanes can leave the load layout (then every later exchange is wave-local)
  static constexpr bool kWave = TT <= 64 && num_passes(N, R) >= 2;
  static constexpr int LSZ = kWave ? N + N / R + col_pad<E, C>() : Padded<N, R>::size;
  static_assert(C * LSZ <= lds_elems<BLOCK, R>(), "LDS array");
  using View = std::conditional_t<kWave, LdsRow<E>, LdsStrided<E, C>>;
  using Sync = std::conditional_t<kWave, WaveSync, BlockSync>;

  __device__ __forceinline__ static size_t table_offset(CMember& m, int step) {
    return (m.pot_expr_len > 0 && (step & 1)) ? size_t(m.X) * size_t(m.P) : 0;
  }
  // potential step multiplier of time index `step` (expPotential; GP phase optional),
  // times the real factor `scale` (the 1/N of the inverse transform that follows).
  // A member with an expression program reads slot step % 2 of its two [P][X] tables
  // (expr_table_kernel fills them before the sweep).
  __device__ __forceinline__ static void potential(cplx<T> (&v)[R], const SweepArgs& a,
                                                   CMember& m, int t_in, int col_in, int step,
                                                   double scale) {
    // opaque lane indices: recomputing theta and x -/+ hbar theta/2 per call is cheaper
    // than keeping them live across the transforms between two calls
    const int t = opaque_v(t_in), col = opaque_v(col_in);
    const double x = m.dx * double(fidx(col, m.X));
    const int row = step < m.pot_rows ? step : m.pot_rows - 1;
    const cptr<double> cf = cmem(m.pot) + size_t(row) * (kMaxDeg + 1);
    const double mask = (m.xmask ? gmem(m.xmask)[col] : 1.0) * scale;
    const bool gp = (a.flags & kGP) != 0;
    const BoppOdd bopp = bopp_odd(cf, m.pot_deg, x, a.vphase);
    // uniform conditions outside the element loops, so that each loop is one basic block
    // and no per-element array stays live across it
    const double hd = a.hbar_half * m.dtheta;
    auto mult = [&](int i) { return expmi(mask, bopp(hd * double(fidx(i, N)))); };
    if (kWave && m.pot_deg >= 0 && !gp) {
      // theta_{N-i} = -theta_i and the phase is odd in u, so the multiplier of N - i is the
      // exact conjugate of that of i (the reduction and the odd/even series negate exactly):
      // lane t evaluates j < R/2 (i < N/2) and takes j >= R/2 from lane TT - t of its team
      // (element R-1-j there); lane 0 pairs with itself (element R-j) and evaluates the
      // self-paired i = N/2 directly.
      cplx<double> M[R / 2];
#pragma unroll
      for (int j = 0; j < R / 2; ++j) M[j] = mult(t + j * TT);
      const cplx<double> nyq = mult(N / 2);
      const int lane = threadIdx.x & 63;
      const int src = lane - t + ((TT - t) & (TT - 1));
      static_for<R / 2, R>([&](auto J) {
        constexpr int j = decltype(J)::value;
        cplx<double> q{__shfl(M[R - 1 - j].x, src, 64), __shfl(M[R - 1 - j].y, src, 64)};
        if constexpr (j == R / 2) {
          if (t == 0) q = {nyq.x, -nyq.y};  // own multiplier (conjugated back below)
        } else {
          if (t == 0) q = M[R - j];
        }
        v[j] = apply(v[j], cplx<double>{q.x, -q.y});
      });
#pragma unroll
      for (int j = 0; j < R / 2; ++j) v[j] = apply(v[j], M[j]);
    } else if (m.pot_deg >= 0 && !gp) {
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = apply(v[j], mult(t + j * TT));
    } else {
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int i = t + j * TT;
        double phi;
        if (m.pot_deg >= 0) {
          phi = bopp(hd * double(fidx(i, N)));
        } else {
          const size_t toff = table_offset(m, step);
          phi = a.vphase * gmem(m.pot_dv)[toff + size_t(i) * m.X + col];
        }
        if (gp) phi -= a.gp_phase * gmem(m.G)[size_t(i) * m.X + col];
        v[j] = apply(v[j], expmi(mask, phi));
      }
    }
  }

  // The same multipliers evaluated apart from their use: they do not depend on the state, so the
  // sweep evaluates them while its loads are in flight (everything but a table and a
  // Gross-Pitaevskii grid together).  Vector loads return in order, so the values that they are
  // made of are loaded before the state: the mask and V's table or the grid G.
  struct MulLoads {
    double mask, tab[R];
  };
  __device__ __forceinline__ static bool early(const SweepArgs& a, CMember& m) {
    return m.pot_deg >= 0 || !(a.flags & kGP);
  }
  __device__ __forceinline__ static void mul_loads(MulLoads& l, const SweepArgs& a, CMember& m, int t, int col,
                                                   int step) {
    l.mask = 1.0;
    if (m.xmask) l.mask = gmem(m.xmask)[col];
    if (m.pot_deg < 0 || (a.flags & kGP)) {
      const size_t toff = m.pot_deg < 0 ? table_offset(m, step) : 0;
      const gptr<const double> src = gmem(m.pot_deg < 0 ? m.pot_dv : const_cast<const double*>(m.G)) + toff;
#pragma unroll
      for (int j = 0; j < R; ++j) l.tab[j] = src[size_t(t + j * TT) * m.X + col];
    }
  }
  __device__ __forceinline__ static void multipliers(cplx<double> (&M)[R], const MulLoads& l, const SweepArgs& a,
                                                     CMember& m, int t, int col, int step, double scale) {
    const double x = m.dx * double(fidx(col, m.X));
    const int row = step < m.pot_rows ? step : m.pot_rows - 1;
    const bool gp = (a.flags & kGP) != 0;
    const double mask = l.mask * scale;
    const BoppOdd bopp = bopp_odd(cmem(m.pot) + size_t(row) * (kMaxDeg + 1), m.pot_deg, x, a.vphase);
    const double hd = a.hbar_half * m.dtheta;
    auto phase = [&](int i) { return bopp(hd * double(fidx(i, N))); };
    if (kWave && m.pot_deg >= 0 && !gp) {
#pragma unroll
      for (int j = 0; j < R / 2; ++j) M[j] = expmi(mask, phase(t + j * TT));
      const cplx<double> nyq = expmi(mask, phase(N / 2));
      const int lane = threadIdx.x & 63;
      const int src = lane - t + ((TT - t) & (TT - 1));
      static_for<R / 2, R>([&](auto J) {
        constexpr int j = decltype(J)::value;
        cplx<double> q{__shfl(M[R - 1 - j].x, src, 64), __shfl(M[R - 1 - j].y, src, 64)};
        if constexpr (j == R / 2) {
          if (t == 0) q = {nyq.x, -nyq.y};
        } else {
          if (t == 0) q = M[R - j];
        }
        M[j] = {q.x, -q.y};
      });
    } else if (m.pot_deg < 0) {
#pragma unroll
      for (int j = 0; j < R; ++j) M[j] = expmi(mask, a.vphase * l.tab[j]);
    } else {
#pragma unroll
      for (int j = 0; j < R; ++j) {
        double phi = phase(t + j * TT);
        if (gp) phi -= a.gp_phase * l.tab[j];
        M[j] = expmi(mask, phi);
      }
    }
  }
  // whether time index step + 1 has the multipliers of step: one row of coefficients, or one
  // table, for both (the merged half steps, which have no Gross-Pitaevskii phase)
  __device__ __forceinline__ static bool same_multipliers(CMember& m, int step) {
    return m.pot_deg >= 0 ? step >= m.pot_rows - 1 : m.pot_expr_len == 0;
  }
  __device__ __forceinline__ static void multiply(cplx<T> (&v)[R], const cplx<double> (&M)[R]) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = apply(v[j], M[j]);
  }

  // The friction operator's factors of this lane's elements: sigma, and theta / N (the 1/N of the
  // inverse transform is a power of two: exact).  REGS: read once per sweep.
  template <bool REGS>
  struct Friction {
    T sg[REGS ? R : 1], th[REGS ? R : 1];
    gptr<const double> sigma, theta;
    __device__ __forceinline__ void load(CMember& m, int t) {
      sigma = gmem(m.sigma_p);
      theta = gmem(m.theta_host);
      if constexpr (REGS) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
          sg[j] = T(sigma[t + j * TT]);
          th[j] = T(theta[t + j * TT] * (1.0 / N));
        }
      }
    }
    __device__ __forceinline__ void by_sigma(cplx<T> (&y)[R], int t) const {
#pragma unroll
      for (int j = 0; j < R; ++j) y[j] = cscale(y[j], REGS ? sg[REGS ? j : 0] : T(sigma[t + j * TT]));
    }
    __device__ __forceinline__ void by_theta(cplx<T> (&y)[R], int t) const {
#pragma unroll
      for (int j = 0; j < R; ++j) y[j] = cscale(y[j], REGS ? th[REGS ? j : 0] : T(theta[t + j * TT] * (1.0 / N)));
    }
  };
  // D(Y) = F_p^{-1}[ theta * F_p[ sigma(p) Y ] ]   (Theta_fp_Damping, FFT.py:1135-1143)
  template <class F, class Tw>
  __device__ __forceinline__ static void cl_operator(cplx<T> (&y)[R], const F& f, int t, View view, const Tw& tw) {
    f.by_sigma(y, t);
    team_fft<T, N, R, -1, View, Sync>(y, t, view, tw);
    f.by_theta(y, t);
    team_fft<T, N, R, +1, View, Sync>(y, t, view, tw);
  }
};

// LDS bytes past the transform arrays of a p-sweep block: per-column sums, then the
// per-column observable terms (<= 64 columns)
constexpr int kPTailBytes = 64 * 12 * 8;
constexpr int kPTailRed = 64 * 11 * 8;  // the last 512 bytes: tile_scale's sums (two per wave)
static_assert(64 * kNCol * 8 <= kPTailRed, "behind the column sums");

// Lanes: the load layout (column cl = tid % C, team index tl = tid / C) makes every
// global load and store instruction cover rows of C consecutive columns.  With wave
// teams the first exchange of the first transform moves each column to one team of
// TT consecutive lanes (column cc = tid / TT, team index tc = tid % TT) and the store
// moves it back through LDS; otherwise the load layout is kept throughout.
template <typename S, typename T, int N, int R, int BLOCK, bool CL, bool TP, typename E>
__device__ __forceinline__ void psweep_body(const SweepArgs& a, CMember& m, int tile,
                                            cplx<E>* lds) {
  using PS = PSweep<T, N, R, BLOCK, E>;
  using View = typename PS::View;
  using Sync = typename PS::Sync;
  constexpr int TT = PS::TT, C = PS::C, LSZ = PS::LSZ;
  constexpr bool kWave = PS::kWave;
  const int tid = threadIdx.x;
  const int cl = tid % C, tl = tid / C;
  const int cc = kWave ? tid / TT : cl, tc = kWave ? tid % TT : tl;
  const int X = m.X;
  const int col = tile * C + cc;
  const gptr<cplx<S>> W = gmem(reinterpret_cast<cplx<S>*>(a.W_dst ? a.W_dst : m.W));
  const Twiddles<T> tw{reinterpret_cast<const cplx<T>*>(m.twP_hi), reinterpret_cast<const cplx<T>*>(m.twP_lo)};
  const View view_c{kWave ? lds + cc * LSZ : lds + cl};
  const int step = (a.flags & kStepArg) ? a.step_add : *cmem(a.step) + a.step_add;

  // 32-bit byte offsets from the member's base (a state is at most 2048^2 x 16 B); the
  // store recomputes them from an opaque copy of the lane index, so that no address
  // stays live (or is spilled) across the transforms
  const unsigned boff = (unsigned(tl) * unsigned(X) + unsigned(tile * C + cl)) * unsigned(sizeof(cplx<S>));
  const unsigned jstride = unsigned(TT) * unsigned(X) * unsigned(sizeof(cplx<S>));
  // radix-8 lanes have the registers to keep the multipliers over the first transform (radix-16
  // lanes spill: -13% on 32 grids of 1024^2)
  constexpr bool kEarly = R <= 8 && !TP;
  // complex128 columns that radix 8 takes from radix 16 (plans of few cells)
  constexpr bool kExact = sizeof(S) == 8 && R == 8 && N >= 1024;
  const bool early = kEarly && PS::early(a, m);
  typename PS::MulLoads ml;
  if (early) PS::mul_loads(ml, a, m, tc, col, step);
  // The friction tables: in registers with the state, or read again for every operator.  Where a CU
  // has one block the wave is alone on its SIMD and the registers are there (FP64, 1024^2: 45.8 us a
  // step, read again 48.4).  Radix-16 lanes in FP32 arithmetic, and the throughput form, run two waves
  // per SIMD only without them (FP32, P = 2048: 214 VGPRs, with them 326; 2048^2 steps: FP32 arithmetic
  // 202 -> 153 us, complex64 states 198 -> 159, complex128 213 -> 174).
  constexpr bool kTabRegs = CL && (R <= 8 || (sizeof(T) == 8 && !TP));
  typename PS::template Friction<kTabRegs> friction;
  double decay[kTabRegs ? R : 1];  // (a plan with friction always has the table)
  if constexpr (CL) friction.load(m, tc);
  if constexpr (kTabRegs && kEarly) {
#pragma unroll
    for (int j = 0; j < R; ++j) decay[j] = gmem(m.theta_decay)[tc + j * TT];
  }
  TilePartials part{0.0, 0.0};
  const bool behind_join = !CL && (a.flags & kTileScale);  // an ODM join's partials give the pending factor
  if (behind_join) part = tile_partials<BLOCK>(a, m);
  ColumnHost host{0.0, 0.0, 0.0};
  if (a.flags & kTilePart) host = column_host(m, tile * C + tid % C);
  cplx<T> v[R];
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = to_arith<T>(gload(at_off(W, boff + unsigned(j) * jstride)));
  const auto twsrc = [&]() {
    if constexpr (kWave && !TP) {
      TwRegs<T, N, R> r;
      load_twiddles<T, N, R>(r, tc, tw);
      return r;
    } else {
      return TwMem<T, kExact>{tw};
    }
  }();
  cplx<double> M[R];
  if (early) PS::multipliers(M, ml, a, m, tc, col, step, 1.0 / N);
  if (a.flags & kScaleOnLoad) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = scale_load(v[j], m.scale);
  }
  if constexpr (kWave) {
    team_fft_remap<T, N, R, -1>(v, tl, LdsRow<E>{lds + cl * LSZ}, tc, view_c, twsrc);
  } else {
    team_fft<T, N, R, -1, View, Sync>(v, tc, view_c, twsrc);
  }
  const auto theta_decay = [&]() {
    if constexpr (kTabRegs) {
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = apply(v[j], cplx<double>{decay[j], 0.0});
    } else if (m.theta_decay) {
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = apply(v[j], cplx<double>{gmem(m.theta_decay)[tc + j * TT], 0.0});
    }
  };
  if (behind_join) {
    const cplx<double> f = tile_scale<BLOCK>(
        a, m, part, reinterpret_cast<double*>(reinterpret_cast<char*>(lds + lds_elems<BLOCK, R>()) + kPTailRed));
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = apply(v[j], f);
  }
  if constexpr (kTabRegs && !kEarly) {  // in flight while potential() evaluates its multipliers
    const int t = opaque_v(tc);
#pragma unroll
    for (int j = 0; j < R; ++j) decay[j] = gmem(m.theta_decay)[t + j * TT];
  }
  if (early)
    PS::multiply(v, M);
  else
    PS::potential(v, a, m, tc, col, step, 1.0 / N);
  theta_decay();
  team_fft<T, N, R, +1, View, Sync>(v, tc, view_c, twsrc);

  if constexpr (CL) {
    // W + 2aD W + (10/3)a^2 D^2 W + (4/3)a^3 D^3 W, a = i dt gamma: the reference's nested
    // LW = W + (2/3)a D W; LW += a D LW; W += 2a D LW (FFT.py:1145-1157) as the sum of the
    // powers, which needs two copies of the column in registers instead of three
    cplx<T> d[R];
#pragma unroll
    for (int j = 0; j < R; ++j) d[j] = v[j];
    const T c1 = T(2.0 * a.cl_a), c2 = T((-10.0 / 3.0) * a.cl_a * a.cl_a),
            c3 = T((-4.0 / 3.0) * a.cl_a * a.cl_a * a.cl_a);
    PS::cl_operator(d, friction, tc, view_c, twsrc);
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = cadd(v[j], mul_i(d[j], c1));
    PS::cl_operator(d, friction, tc, view_c, twsrc);
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = cadd(v[j], cscale(d[j], c2));
    PS::cl_operator(d, friction, tc, view_c, twsrc);
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = cadd(v[j], mul_i(d[j], c3));
  }

  // per-column sums of the tile in the LDS tail: csum[c * kNCol + k] for column tile*C + c
  double* csum = reinterpret_cast<double*>(reinterpret_cast<char*>(lds) + lds_elems<BLOCK, R>() * sizeof(cplx<E>));
  // column sums to global memory, after a block barrier that follows their LDS write
  const auto publish_colsums = [&]() {
    if (tid < C) {
#pragma unroll
      for (int k = 0; k < kNCol; ++k) gmem(m.colsums)[size_t(tile * C + tid) * kNCol + k] = csum[tid * kNCol + k];
    }
  };
  bool colsums_pending = false;
  if (a.flags & kColSums) {
    double acc[kNCol] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const double p = gmem(m.p_host)[tc + j * TT];
      const double w = double(v[j].x);
      acc[0] += w;
      acc[1] += double(v[j].y);
      acc[2] += p * w;
      acc[3] += p * p * w;
      acc[4] += w < 0.0 ? w : 0.0;
    }
    if constexpr (kWave) {
      // a column's lanes are TT consecutive lanes of one wave; the last one gets the sums
#pragma unroll
      for (int k = 0; k < kNCol; ++k) acc[k] = group_sum<TT>(acc[k]);
      if (tc == TT - 1) {
#pragma unroll
        for (int k = 0; k < kNCol; ++k) csum[cc * kNCol + k] = acc[k];
      }
      if (a.flags & kMerge) {
        __syncthreads();
        publish_colsums();
      } else {
        colsums_pending = true;  // published after the store's block barrier
      }
    } else {
      // lanes of one column inside a wave: c + C*t; fold t with xor shuffles
#pragma unroll
      for (int off = C; off < 64; off <<= 1) {
#pragma unroll
        for (int k = 0; k < kNCol; ++k) acc[k] += __shfl_xor(acc[k], off, 64);
      }
      constexpr int kWaves = (BLOCK + 63) / 64;
      constexpr int kLanes = C < 64 ? C : 64;  // distinct columns per wave
      __syncthreads();
      double* red = reinterpret_cast<double*>(lds);
      const int wave = tid >> 6, lane = tid & 63;
      if (lane < kLanes) {
#pragma unroll
        for (int k = 0; k < kNCol; ++k) red[(wave * kLanes + lane) * kNCol + k] = acc[k];
      }
      __syncthreads();
      if (tid < C) {
        // C <= 64: every wave holds all C columns
        double sc[kNCol] = {0.0, 0.0, 0.0, 0.0, 0.0};
        for (int w = 0; w < kWaves; ++w) {
#pragma unroll
          for (int k = 0; k < kNCol; ++k) sc[k] += red[(w * kLanes + tid) * kNCol + k];
        }
#pragma unroll
        for (int k = 0; k < kNCol; ++k) {
          gmem(m.colsums)[size_t(tile * C + tid) * kNCol + k] = sc[k];
          csum[tid * kNCol + k] = sc[k];
        }
      }
      __syncthreads();  // csum complete for the tile partials; red free for the transforms
    }
  }

  if (a.flags & kMerge) {
    if (early && !PS::same_multipliers(m, step)) {
      const int t = opaque_v(tc), c = opaque_v(col);
      PS::mul_loads(ml, a, m, t, c, step + 1);
      PS::multipliers(M, ml, a, m, t, c, step + 1, 1.0 / N);
    }
    team_fft<T, N, R, -1, View, Sync>(v, tc, view_c, twsrc);
    if (early)
      PS::multiply(v, M);
    else
      PS::potential(v, a, m, tc, col, step + 1, 1.0 / N);
    theta_decay();
    team_fft<T, N, R, +1, View, Sync>(v, tc, view_c, twsrc);
  }

  if constexpr (kWave) {
    // back to the load layout: natural order through the team's LDS array
    Sync::sync();
#pragma unroll
    for (int j = 0; j < R; ++j) *view_c.ptr(padr<R>(tc + j * TT)) = ccvt<E>(v[j]);
    __syncthreads();
    if (colsums_pending) publish_colsums();
    const LdsRow<E> view_l{lds + cl * LSZ};
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = ccvt<T>(*view_l.ptr(padr<R>(tl + j * TT)));
  }
  const int ts = opaque_v(int(threadIdx.x));  // offset recomputed from the lane index
  const unsigned soff = (unsigned(ts / C) * unsigned(X) + unsigned(tile * C + ts % C)) * unsigned(sizeof(cplx<S>));
#pragma unroll
  for (int j = 0; j < R; ++j) store_cached(at_off(W, soff + unsigned(j) * jstride), to_arith<S>(v[j]));
  if (a.flags & kTilePart) write_tile_partial<C>(a, m, tile, csum, host, step - a.step_add);
  if ((a.flags & kRecStep) && tid == 0 && tile == 0 && first_member(a, m)) *gmem(a.rec_step) = step - a.step_add;
}

// ------------------------------------------------------------------ Gross-Pitaevskii shift
// One theta row of G per team from the density rho(t + j TT) held in v (real parts).
template <int N, int R, int BLOCK, class M>
__device__ __forceinline__ void gpshift_rows(cplx<double> (&v)[R], const M& m, int tile, cplx<double>* lds) {
  constexpr int TT = N / R, ROWS = BLOCK / TT;
  constexpr int LSZ = Padded<N, R>::size;
  using Sync = std::conditional_t<(TT <= 64), WaveSync, BlockSync>;
  const int tid = threadIdx.x, team = tid / TT, t = tid % TT;
  const int row = tile * ROWS + team;
  const Twiddles<double> tw{reinterpret_cast<const cplx<double>*>(m.twX64), nullptr};
  LdsRow<double> view{lds + team * LSZ};
  // the multiplier does not depend on the density: evaluated while its loads are in flight
  double f[R];
  const double half_theta = 0.5 * cmem(m.theta_host)[row];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    double cs;
    sincos_fp64(gmem(m.lambda_host)[t + j * TT] * half_theta, &f[j], &cs);
  }
  const auto twsrc = [&]() {
    if constexpr (TT <= 64) {
      TwRegs<double, N, R> r;
      load_twiddles<double, N, R>(r, t, tw);
      return r;
    } else {
      return TwMem<double>{tw};
    }
  }();
  team_fft<double, N, R, -1, LdsRow<double>, Sync>(v, t, view, twsrc);
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = {2.0 * f[j] * v[j].y, -2.0 * f[j] * v[j].x};  // (-2i sin) (a + ib)
  team_fft<double, N, R, +1, LdsRow<double>, Sync>(v, t, view, twsrc);
#pragma unroll
  for (int j = 0; j < R; ++j) gmem(m.G)[size_t(row) * N + t + j * TT] = v[j].x * (1.0 / N);
}

// kTileScale: the state is that of the p sweep just done: its density is the column sums times the
// pending factor (from the tile partials, as in the x sweep), and the member's record item forms
// the record row; without it the density is read from m.rho.  kProbSq: tile 0 records
// dX sum rho^2 (GP.py:1937-1939).
template <int N, int R, int BLOCK>
__device__ __forceinline__ void gpshift_body(const SweepArgs& a, CMember& m, int tile, cplx<double>* lds) {
  constexpr int TT = N / R;
  const int t = threadIdx.x % TT;
  cplx<double> v[R];
  if (a.flags & kTileScale) {
    const TilePartials part = tile_partials<BLOCK>(a, m);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const gptr<const double> cs = gmem(const_cast<const double*>(m.colsums)) + size_t(t + j * TT) * kNCol;
      v[j] = {cs[0], cs[1]};
    }
    const cplx<double> f = tile_scale<BLOCK>(a, m, part, reinterpret_cast<double*>(lds + lds_elems<BLOCK, R>()));
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = {(v[j].x * f.x - v[j].y * f.y) * m.rho_factor, 0.0};
  } else {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = {gmem(m.rho)[t + j * TT], 0.0};
  }
  if ((a.flags & kProbSq) && tile == 0) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j) s = fma(v[j].x, v[j].x, s);
    constexpr int G = TT < 64 ? TT : 64;
    s = group_sum<G>(s);  // of one team, or of each of a team's waves
    if constexpr (TT > 64) {
      double* red = reinterpret_cast<double*>(lds + lds_elems<BLOCK, R>());
      if (threadIdx.x % 64 == 63) red[threadIdx.x / 64] = s;
      __syncthreads();
      s = 0.0;
#pragma unroll
      for (int w = 0; w < TT / 64; ++w) s += red[w];
    }
    if (threadIdx.x == TT - 1) gmem(m.obs)[size_t(*cmem(a.step) - m.obs_base) * kNObs + kObsProbSq] = m.dx_host * s;
  }
  gpshift_rows<N, R, BLOCK>(v, m, tile, lds);
}

// ------------------------------------------------------------------ kernels
// sizes up to MAXN.  One launch covers members of every size: the throughput forms (sides
// up to 1024) spill a few VGPRs at three waves per SIMD, in the general-polynomial kinetic
// branch, and still run an uneven 128..1024 ensemble 2% faster than one launch per size
// (and a uniform batch within 0.5%)
#define WH_DISPATCH_TO(NVAR, BODY, MAXN)                                                     \
  switch (NVAR) {                                                                            \
    case 128: if constexpr (size_ok<128, R, BLOCK>() && 128 <= (MAXN)) { BODY(128); } break;   \
    case 256: if constexpr (size_ok<256, R, BLOCK>() && 256 <= (MAXN)) { BODY(256); } break;   \
    case 512: if constexpr (size_ok<512, R, BLOCK>() && 512 <= (MAXN)) { BODY(512); } break;   \
    case 1024: if constexpr (size_ok<1024, R, BLOCK>() && 1024 <= (MAXN)) { BODY(1024); } break; \
    case 2048: if constexpr (size_ok<2048, R, BLOCK>() && 2048 <= (MAXN)) { BODY(2048); } break; \
    default: break;                                                                          \
  }
#define WH_DISPATCH(NVAR, BODY) WH_DISPATCH_TO(NVAR, BODY, 2048)

// Two waves per SIMD (<= 256 VGPRs) for the plain sweeps: a batch of grids overlaps one
// wave's loads and stores with the other's transforms; three for the throughput form
// (TP: table twiddles, exchanges in the storage precision).  The Caldeira-Leggett p sweep holds
// two state copies: its plain forms may take the full register file of one wave, its throughput
// form fits two, and exchanges in the arithmetic precision there (rounding the exchanges to
// complex64 gains nothing: 2048^2 161 us a step in FP64, 162 rounded).
template <typename S, typename T, bool TP>
using LdsElem = std::conditional_t<TP, S, T>;
template <typename S, typename T, int R, int BLOCK, bool TP>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(TP ? 3 : 2))) xsweep_kernel(SweepArgs a) {
  using E = LdsElem<S, T, TP>;
  __shared__ cplx<E> lds[lds_elems<BLOCK, R>() + kTileRedBytes / sizeof(cplx<E>)];
  const unsigned w = x_item(a);
  CMember& m = member_at(a.members, w >> 16);
  // the fields that the sweep's loads wait for, in one round of scalar loads (left to its use, each
  // came after a wait of its own: 1024^2 x sweep 15.9 -> 14.7 us, p sweep with friction 32.2 -> 30.6)
  asm volatile("" ::"s"(m.W), "s"(m.X), "s"(m.P), "s"(m.twX_hi), "s"(m.tilepart), "s"(m.dp), "s"(m.dlambda),
               "s"(m.dxdp), "s"(m.scale), "s"(m.lambda_decay));
  const int tile = int(w & 0xffffu);
  if (tile == kRecordTile) {
    if (a.flags & kTileScale) record_item<BLOCK>(a, m, reinterpret_cast<double*>(lds));
    return;
  }
#define BODY(n) xsweep_body<S, T, n, R, BLOCK, TP, E>(a, m, tile, lds)
  WH_DISPATCH_TO(m.X, BODY, TP ? kTpMaxN : 2048)
#undef BODY
}

template <typename S, typename T, int R, int BLOCK, bool CL, bool TP>
__device__ __forceinline__ void psweep_entry(const SweepArgs& a) {
  using E = LdsElem<S, T, TP && !CL>;
  __shared__ cplx<E> lds[lds_elems<BLOCK, R>() + kPTailBytes / sizeof(cplx<E>)];
  const unsigned w = p_item(a);
  CMember& m = member_at(a.members, w >> 16);
  // the fields that the sweep's loads wait for, in one round of scalar loads
  asm volatile("" ::"s"(m.W), "s"(m.X), "s"(m.P), "s"(m.pot), "s"(m.pot_deg), "s"(m.pot_rows), "s"(m.xmask),
               "s"(m.theta_decay), "s"(m.twP_hi), "s"(m.x_host), "s"(m.dv_host), "s"(m.v0_host), "s"(m.p_host),
               "s"(m.dx), "s"(m.dtheta), "s"(m.sigma_p), "s"(m.theta_host), "s"(*cmem(a.step)));
  const int tile = int(w & 0xffffu);
#define BODY(n) psweep_body<S, T, n, R, BLOCK, CL, TP, E>(a, m, tile, lds)
  WH_DISPATCH_TO(m.P, BODY, TP && !CL ? kTpMaxN : 2048)
#undef BODY
}
template <typename S, typename T, int R, int BLOCK, bool CL, bool TP>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(CL ? 1 : TP ? 3 : 2))) psweep_kernel(SweepArgs a) {
  psweep_entry<S, T, R, BLOCK, CL, TP>(a);
}

template <int R, int BLOCK>
__global__ void __launch_bounds__(BLOCK) gpshift_kernel(SweepArgs a) {
  __shared__ cplx<double> lds[lds_elems<BLOCK, R>() + kTileRedBytes / sizeof(cplx<double>)];
  const unsigned w = x_item(a);
  CMember& m = member_at(a.members, w >> 16);
  const int tile = int(w & 0xffffu);
  asm volatile("" ::"s"(m.X), "s"(m.P), "s"(m.rho), "s"(m.colsums), "s"(m.tilepart), "s"(m.G), "s"(m.twX64),
               "s"(m.lambda_host), "s"(m.theta_host), "s"(m.rho_factor), "s"(m.dxdp));
  if (tile == kRecordTile) {
    if (a.flags & kTileScale) record_item<BLOCK>(a, m, reinterpret_cast<double*>(lds));
    return;
  }
#define BODY(n) gpshift_body<n, R, BLOCK>(a, m, tile, lds)
  WH_DISPATCH(m.X, BODY)
#undef BODY
}

}  // namespace wh
