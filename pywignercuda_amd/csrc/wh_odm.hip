// ODM Lindblad dissipator of GPU_Wigner2D_FFT (dampingFunction = 'ODM', order 1:
// W += L(W), Lindbladian_ODM_Order1 -> _Lindbladian_ODM, GPU_Wigner2D_FFT.py:1516-1634,
// 1907-1910; tables of SetA_ODM, :1196-1244).
//
// The reference sums six terms h_k(theta, x) F_p F_x^-1 [g_k(p, lambda) F_x W] (18 FFTs).
// With c+- = cos(x +- hbar theta/2), s+- = sin(x +- hbar theta/2) the products of its h_k
// split into functions of x alone and of theta alone:
//   c+c- = (cos 2x + cos hbar theta)/2,  s+s- = (cos hbar theta - cos 2x)/2,
//   c-s+ = (sin 2x + sin hbar theta)/2,  s-c+ = (sin 2x - sin hbar theta)/2,
// an x factor commutes with F_p and a theta factor with F_x, so
//   L(W)/(2 gamma dt) = cos2x/2 F_x^-1[A W^] + i s sin2x/2 F_x^-1[B W^] + F_x^-1[C W^]
//                     + F_x^-1 F_p^-1 [ cos(hbar theta)/2 F_p[E W^] + i s sin(hbar theta)/2 F_p[F W^] ]
// with W^ = F_x W, g+- = g(p +- hbar lambda/2), gs+- = sign(p +- hbar lambda/2) g+-,
//   A = g+g- - gs+gs-,  B = g+gs- - gs+g-,  C = -(g+^2 + g-^2)/2,
//   E = g+g- + gs+gs-,  F = g+gs- + gs+g-.
// Three sweeps: odm_x (rows: F_x, the three x terms, W += c Lx, E W^ and F W^ to scratch),
// odm_p (columns of the scratch: F_p, theta factors, F_p^-1) and odm_back (rows: W += F_x^-1);
// between two iterations odm_back also takes the observables and does the next kinetic step.
#include <hip/hip_runtime.h>

#include "wh_fft.hpp"
#include "wh_kernels.hpp"
#include "wh_math.hpp"
#include "wh_sweeps.hpp"

namespace wh {

constexpr int kOdmR = 8;
constexpr int kOdmBlock = 256;

namespace {

template <typename U>
__device__ __forceinline__ cplx<double> wide(cplx<U> v) {
  return {double(v.x), double(v.y)};
}
template <typename U>
__device__ __forceinline__ cplx<U> nar(cplx<double> v) {
  return {U(v.x), U(v.y)};
}

// store of a complex element (one 2-vector store)
template <typename U>
__device__ __forceinline__ void put(gptr<cplx<U>> p, cplx<U> v) {
  store_cached<U>(p, v);
}

}  // namespace

// Order of the loads and registers.  At 512^2 every sweep is one latency after another (one wave
// per SIMD on half of the CUs), so each body issues the loads of its tables before those of the
// state, keeps what it needs again in registers, and has wave teams up to N = 512 (exchanges
// without block barriers, twiddles in registers).
template <int N, int R>
using OdmSync = std::conditional_t<(N / R <= 64), WaveSync, BlockSync>;
template <typename T, int N, int R>
__device__ __forceinline__ auto odm_twiddles(const Twiddles<T>& tw, int t) {
  if constexpr (N / R <= 64) {
    TwRegs<T, N, R> r;
    load_twiddles<T, N, R>(r, t, tw);
    return r;
  } else {
    return TwMem<T>{tw};
  }
}

// weight, sgn: the channel's weight and sign (GPU_Wigner2D_ODM2 runs two channels,
// (weightLindbland1, +1) then (weightLindbland2, -1), GPU_Wigner2D_FFT.py:2173-2181)
template <typename S, typename T, int N, int R, int BLOCK>
__device__ __forceinline__ void odm_x_body(CMember& m, int tile, cplx<T>* lds, double weight, double sgn) {
  constexpr int TT = N / R, ROWS = BLOCK / TT;
  constexpr int LSZ = Padded<N, R>::size;
  const int tid = threadIdx.x, team = tid / TT, t = tid % TT;
  const int row = tile * ROWS + team;
  const unsigned PX = unsigned(m.P) * unsigned(N), e0 = unsigned(row) * unsigned(N) + unsigned(t);
  const gptr<cplx<S>> W = gmem(reinterpret_cast<cplx<S>*>(m.W)) + e0;
  const gptr<cplx<T>> S1 = gmem(reinterpret_cast<cplx<T>*>(m.odm_s)) + e0;
  const gptr<const double> g = gmem(const_cast<const double*>(m.odm_g)) + e0;
  const Twiddles<T> tw{reinterpret_cast<const cplx<T>*>(m.twX_hi), reinterpret_cast<const cplx<T>*>(m.twX_lo)};
  LdsRow<T> view{lds + team * LSZ};
  using Sync = OdmSync<N, R>;

  double gp[R], gm[R], gsp[R], gsm[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    gp[j] = g[j * TT];
    gm[j] = g[size_t(PX) + j * TT];
    gsp[j] = g[2 * size_t(PX) + j * TT];
    gsm[j] = g[3 * size_t(PX) + j * TT];
  }
  const auto twsrc = odm_twiddles<T, N, R>(tw, t);
  cplx<T> f[R], w0[R];
#pragma unroll
  for (int j = 0; j < R; ++j) w0[j] = to_arith<T>(gload(W + j * TT));
#pragma unroll
  for (int j = 0; j < R; ++j) f[j] = w0[j];
  team_fft<T, N, R, -1, LdsRow<T>, Sync>(f, t, view, twsrc);  // W^ = F_x W
  // theta terms' inputs E W^, F W^ (lambda picture)
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const cplx<double> w = wide(f[j]);
    const double E = gp[j] * gm[j] + gsp[j] * gsm[j], F = gp[j] * gsm[j] + gsp[j] * gm[j];
    put(S1 + j * TT, nar<T>({E * w.x, E * w.y}));
    put(S1 + size_t(PX) + j * TT, nar<T>({F * w.x, F * w.y}));
  }
  // x terms
  cplx<double> acc[R];
  const double inv = 1.0 / N;
#pragma unroll
  for (int term = 0; term < 3; ++term) {
    cplx<T> y[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const double k = term == 0   ? gp[j] * gm[j] - gsp[j] * gsm[j]
                       : term == 1 ? gp[j] * gsm[j] - gsp[j] * gm[j]
                                   : -0.5 * (gp[j] * gp[j] + gm[j] * gm[j]);
      y[j] = nar<T>({k * double(f[j].x), k * double(f[j].y)});
    }
    double h[R];
    if (term < 2) {
#pragma unroll
      for (int j = 0; j < R; ++j) h[j] = gmem(m.odm_x)[(term ? N : 0) + t + j * TT];
    }
    team_fft<T, N, R, +1, LdsRow<T>, Sync>(y, t, view, twsrc);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const cplx<double> u = wide(y[j]);
      if (term == 0) {
        const double c = 0.5 * h[j] * inv;  // cos 2x / 2
        acc[j] = {c * u.x, c * u.y};
      } else if (term == 1) {
        const double c = 0.5 * m.odm_sign * sgn * h[j] * inv;  // i s sin 2x / 2
        acc[j] = {acc[j].x - c * u.y, acc[j].y + c * u.x};
      } else {
        acc[j] = {acc[j].x + inv * u.x, acc[j].y + inv * u.y};
      }
    }
  }
  const double c = m.odm_c * weight;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const cplx<double> w = wide(w0[j]);
    put(W + j * TT, nar<S>({w.x + c * acc[j].x, w.y + c * acc[j].y}));
  }
}

// Columns of the scratch in the load layout, moved to wave teams at the first exchange and back
// for the store, as the p sweep does (PSweep); two transforms share the LDS array.
template <typename S, typename T, int N, int R, int BLOCK>
__device__ __forceinline__ void odm_p_body(CMember& m, int tile, cplx<T>* lds, double weight, double sgn) {
  using PS = PSweep<T, N, R, BLOCK>;
  using View = typename PS::View;
  using Sync = typename PS::Sync;
  constexpr int TT = PS::TT, C = PS::C, LSZ = PS::LSZ;
  constexpr bool kWave = PS::kWave;
  const int tid = threadIdx.x;
  const int cl = tid % C, tl = tid / C;
  const int cc = kWave ? tid / TT : cl, tc = kWave ? tid % TT : tl;
  const int X = m.X;
  const unsigned PX = unsigned(N) * unsigned(X);
  const gptr<cplx<T>> S1 = gmem(reinterpret_cast<cplx<T>*>(m.odm_s));
  const Twiddles<T> tw{reinterpret_cast<const cplx<T>*>(m.twP_hi), reinterpret_cast<const cplx<T>*>(m.twP_lo)};
  const View view_c{kWave ? lds + cc * LSZ : lds + cl};
  const unsigned e0 = unsigned(tl) * unsigned(X) + unsigned(tile * C + cl), stride = unsigned(TT) * unsigned(X);
  double ct[R], st[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    ct[j] = gmem(m.odm_th)[tc + j * TT];
    st[j] = gmem(m.odm_th)[N + tc + j * TT];
  }
  const auto twsrc = odm_twiddles<T, N, R>(tw, tc);
  cplx<T> a[R], b[R];
#pragma unroll
  for (int j = 0; j < R; ++j) a[j] = gload(S1 + (e0 + unsigned(j) * stride));
#pragma unroll
  for (int j = 0; j < R; ++j) b[j] = gload(S1 + (size_t(PX) + e0 + unsigned(j) * stride));
  if constexpr (kWave) {
    const LdsRow<T> view_l{lds + cl * LSZ};
    team_fft_remap<T, N, R, -1>(a, tl, view_l, tc, view_c, twsrc);
    __syncthreads();  // the columns' arrays are free for the other transform's lanes
    team_fft_remap<T, N, R, -1>(b, tl, view_l, tc, view_c, twsrc);
  } else {
    team_fft<T, N, R, -1, View, Sync>(a, tc, view_c, twsrc);
    team_fft<T, N, R, -1, View, Sync>(b, tc, view_c, twsrc);
  }
  const double k = 0.5 * m.odm_c * weight / N, s = m.odm_sign * sgn;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const cplx<double> ua = wide(a[j]), ub = wide(b[j]);
    // (c/2) [cos(hbar theta) a + i s sin(hbar theta) b] / P
    a[j] = nar<T>({k * (ct[j] * ua.x - s * st[j] * ub.y), k * (ct[j] * ua.y + s * st[j] * ub.x)});
  }
  team_fft<T, N, R, +1, View, Sync>(a, tc, view_c, twsrc);
  if constexpr (kWave) {
    Sync::sync();
#pragma unroll
    for (int j = 0; j < R; ++j) *view_c.ptr(padr<R>(tc + j * TT)) = a[j];
    __syncthreads();
    const LdsRow<T> view_l{lds + cl * LSZ};
#pragma unroll
    for (int j = 0; j < R; ++j) a[j] = *view_l.ptr(padr<R>(tl + j * TT));
  }
#pragma unroll
  for (int j = 0; j < R; ++j) put(S1 + (e0 + unsigned(j) * stride), a[j]);
}

// W += F_x^-1 of the scratch.  JOIN: the last sweep of an iteration and the first of the next in
// one launch: the observables of the new state (each tile its 12 partial sums, as a p sweep's
// tile writes them; an item of the next odm_x launch forms the record) and, in the Lie scheme
// (KIN), the next kinetic step on the row that is in registers.  The renormalisation factor
// needs all rows: the next p sweep applies it (kTileScale).
template <typename S, typename T, int N, int R, int BLOCK, bool JOIN>
__device__ __forceinline__ void odm_back_body(const SweepArgs& a, CMember& m, int tile, cplx<T>* lds) {
  constexpr int TT = N / R, ROWS = BLOCK / TT;
  constexpr int LSZ = Padded<N, R>::size;
  const int tid = threadIdx.x, team = tid / TT, t = tid % TT;
  const int row = tile * ROWS + team;
  const unsigned e0 = unsigned(row) * unsigned(N) + unsigned(t);
  const gptr<cplx<S>> W = gmem(reinterpret_cast<cplx<S>*>(m.W)) + e0;
  const gptr<const cplx<T>> S1 = gmem(reinterpret_cast<const cplx<T>*>(m.odm_s)) + e0;
  const Twiddles<T> tw{reinterpret_cast<const cplx<T>*>(m.twX_hi), reinterpret_cast<const cplx<T>*>(m.twX_lo)};
  LdsRow<T> view{lds + team * LSZ};
  using Sync = OdmSync<N, R>;
  cplx<T> y[R], w0[R];
#pragma unroll
  for (int j = 0; j < R; ++j) y[j] = gload<T>(S1 + j * TT);
#pragma unroll
  for (int j = 0; j < R; ++j) w0[j] = to_arith<T>(gload(W + j * TT));
  const auto twsrc = odm_twiddles<T, N, R>(tw, t);
  ColumnHost host[JOIN ? R : 1];
  double ph = 0.0;
  if constexpr (JOIN) {
#pragma unroll
    for (int j = 0; j < R; ++j) host[j] = column_host(m, t + j * TT);
    ph = gmem(m.p_host)[row];
  }
  team_fft<T, N, R, +1, LdsRow<T>, Sync>(y, t, view, twsrc);
  const double inv = 1.0 / N;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const cplx<double> w = wide(w0[j]), u = wide(y[j]);
    w0[j] = to_arith<T>(nar<S>({w.x + inv * u.x, w.y + inv * u.y}));  // the state as it is stored
  }
  if constexpr (JOIN) {
    // the row's sums over x, then the terms with p
    double s0 = 0.0, si = 0.0, sx = 0.0, sxx = 0.0, sdv = 0.0, sxdv = 0.0, sv = 0.0, sn = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const double w = double(w0[j].x);
      s0 += w;
      si += double(w0[j].y);
      sx = fma(host[j].x, w, sx);
      sxx = fma(host[j].x * host[j].x, w, sxx);
      sdv = fma(host[j].dv, w, sdv);
      sxdv = fma(host[j].x * host[j].dv, w, sxdv);
      sv = fma(host[j].v0, w, sv);
      sn += w < 0.0 ? w : 0.0;
    }
    double o[12] = {s0, si, sx, sxx, ph * s0, ph * ph * s0, ph * sx, sdv, ph * sdv, sxdv,
                    fma(ph * ph * m.inv_2m, s0, sv), sn};
    double* red = reinterpret_cast<double*>(lds + lds_elems<BLOCK, R>());
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int k = 0; k < 12; ++k) o[k] = group_sum<64>(o[k]);
    if (lane == 63) {
#pragma unroll
      for (int k = 0; k < 12; ++k) red[wave * 12 + k] = o[k];
    }
    if (a.kin_linear) {
      // the Lie kinetic step (lambda dt p / m), as xsweep_body's linear form
      const double ak = a.dt * m.dlambda * (a.k_c0 + a.k_c1 * m.dp * double(fidx(row, m.P)));
      const cplx<double> Et = expmi(inv, ak * double(t)), Z1 = expmi(1.0, ak * double(TT));
      team_fft<T, N, R, -1, LdsRow<T>, Sync>(w0, t, view, twsrc);
      kinetic_apply<T, R, TT>(w0, m, t, Et, Z1);
      team_fft<T, N, R, +1, LdsRow<T>, Sync>(w0, t, view, twsrc);
    }
    __syncthreads();
    if (tid < 12) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < BLOCK / 64; ++w) s += red[w * 12 + tid];
      gmem(m.tilepart)[size_t(tid) * m.X + tile] = s;
    }
    if (tid == 0 && tile == 0 && first_member(a, m)) *gmem(a.step) = *cmem(a.rec_step) + 1;
  }
#pragma unroll
  for (int j = 0; j < R; ++j) put(W + j * TT, to_arith<S>(w0[j]));
}

// KIND: kOdmX, kOdmP, kOdmBack, kOdmJoin.  The list of kOdmX ends with the members' record items; a launch
// that is not to record (no join's partials are there yet, or another channel's did) is cut before them.
template <typename S, typename T, int KIND>
__global__ void __launch_bounds__(kOdmBlock) odm_kernel(SweepArgs a, double weight, double sgn) {
  __shared__ cplx<T> lds[lds_elems<kOdmBlock, kOdmR>() + kTileRedBytes / sizeof(cplx<T>)];
  const unsigned w = x_item(a);
  CMember& m = member_at(a.members, w >> 16);
  const int tile = int(w & 0xffffu);
  asm volatile("" ::"s"(m.W), "s"(m.X), "s"(m.P), "s"(m.odm_s), "s"(m.odm_g), "s"(m.odm_x), "s"(m.odm_th),
               "s"(m.twX_hi), "s"(m.twP_hi), "s"(m.x_host), "s"(m.dv_host), "s"(m.v0_host), "s"(m.p_host));
  constexpr int R = kOdmR, BLOCK = kOdmBlock;
  if constexpr (KIND == kOdmX) {
    if (tile == kRecordTile) {
      record_item<BLOCK, true>(a, m, reinterpret_cast<double*>(lds));
      return;
    }
#define BODY(n) odm_x_body<S, T, n, R, BLOCK>(m, tile, lds, weight, sgn)
    WH_DISPATCH(m.X, BODY)
#undef BODY
  } else if constexpr (KIND == kOdmP) {
#define BODY(n) odm_p_body<S, T, n, R, BLOCK>(m, tile, lds, weight, sgn)
    WH_DISPATCH(m.P, BODY)
#undef BODY
  } else {
#define BODY(n) odm_back_body<S, T, n, R, BLOCK, KIND == kOdmJoin>(a, m, tile, lds)
    WH_DISPATCH(m.X, BODY)
#undef BODY
  }
}

// Tiles of the ODM sweeps for one member: rows per x tile, columns per p tile.
int odm_rows_per_tile(int X) { return kOdmBlock / (X / kOdmR); }
int odm_cols_per_tile(int P) { return kOdmBlock / (P / kOdmR); }
int odm_radix() { return kOdmR; }
int odm_block() { return kOdmBlock; }

template <typename S, typename T>
hipError_t odm_launch(int kind, const SweepArgs& a, int nwork, double weight, double sgn, hipStream_t s) {
  const dim3 g(nwork), b(kOdmBlock);
  switch (kind) {
    case kOdmX: hipLaunchKernelGGL((odm_kernel<S, T, kOdmX>), g, b, 0, s, a, weight, sgn); break;
    case kOdmP: hipLaunchKernelGGL((odm_kernel<S, T, kOdmP>), g, b, 0, s, a, weight, sgn); break;
    case kOdmBack: hipLaunchKernelGGL((odm_kernel<S, T, kOdmBack>), g, b, 0, s, a, weight, sgn); break;
    case kOdmJoin: hipLaunchKernelGGL((odm_kernel<S, T, kOdmJoin>), g, b, 0, s, a, weight, sgn); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_odm(int prec, int kind, const SweepArgs& a, int nwork, double weight, double sgn, hipStream_t s) {
  if (prec == 0) return odm_launch<double, double>(kind, a, nwork, weight, sgn, s);
  if (prec == 1) return odm_launch<float, float>(kind, a, nwork, weight, sgn, s);
  return odm_launch<float, double>(kind, a, nwork, weight, sgn, s);
}

}  // namespace wh
