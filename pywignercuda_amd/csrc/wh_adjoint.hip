// Adjoint (reverse-time) step of the Lie split operator, for gradients of a loss
// of the final state with respect to the polynomial coefficients a_k(n) of V.
//
// Forward step n (GPU_Wigner2D_FFT.py:1884-1899): W_{n+1} = F_p^-1 M_n F_p K W_n,
// M_n = r exp(-i phi_n), phi_n = vphase (V_n(x - u) - V_n(x + u)), u = hbar theta / 2.
// Adjoint state: Lambda_n = U_n^dagger Lambda_{n+1}
//                         = K^dagger F_p^-1 conj(M_n) F_p Lambda_{n+1}
// (p sweep with the conjugated potential multiplier, then the x sweep with the
// conjugated kinetic multiplier).  Gradient (Parseval along p, numpy conventions):
//   dL/da_k(n) = Re sum conj(Lambda_{n+1}) dU_n/da_k W_n
//              = (vphase / P) sum_{theta,x} g_k Im( conj(F_p Lambda_{n+1}) F_p W_{n+1} ),
//   g_k = (x - u)^k - (x + u)^k,
// so the adjoint p sweep reads Lambda_{n+1} and the forward state W_{n+1} and sums
// u^q Im(...) of each column for q = 1, 3, 5, 7, from which
//   g_k = -2 sum_{q odd <= k} C(k, q) x^(k-q) u^q
// gives the nine gradient terms of the column.
#include <hip/hip_runtime.h>

#include "wh_sweeps.hpp"

namespace wh {

// Moments of u per column: q = 1, 3, 5, 7.
constexpr int kAdjMom = (kMaxDeg + 1) / 2;

// Columns in the load layout, moved to wave teams at the first exchange and back for the store, as
// the p sweep does (PSweep).  512^2: 10.9 us; with block barriers around every exchange, two
// polynomials and 18 powers per cell it was 19.7.
template <typename T, int N, int R, int BLOCK>
__device__ __forceinline__ void adj_psweep_body(const SweepArgs& a, CMember& m, int tile, cplx<T>* lds,
                                                const void* W_next, double* gcols) {
  using PS = PSweep<T, N, R, BLOCK>;
  using View = typename PS::View;
  using Sync = typename PS::Sync;
  constexpr int TT = PS::TT, C = PS::C, LSZ = PS::LSZ;
  constexpr bool kWave = PS::kWave;
  const int tid = threadIdx.x;
  const int cl = tid % C, tl = tid / C;
  const int cc = kWave ? tid / TT : cl, tc = kWave ? tid % TT : tl;
  const int X = m.X;
  const int col = tile * C + cc;
  const gptr<cplx<T>> L = gmem(reinterpret_cast<cplx<T>*>(a.W_dst));
  const gptr<const cplx<T>> F = gmem(reinterpret_cast<const cplx<T>*>(W_next));
  const Twiddles<T> tw{reinterpret_cast<const cplx<T>*>(m.twP_hi), reinterpret_cast<const cplx<T>*>(m.twP_lo)};
  const View view_c{kWave ? lds + cc * LSZ : lds + cl};
  const unsigned boff = (unsigned(tl) * unsigned(X) + unsigned(tile * C + cl)) * unsigned(sizeof(cplx<T>));
  const unsigned jstride = unsigned(TT) * unsigned(X) * unsigned(sizeof(cplx<T>));
  const int step = a.step_add;

  typename PS::MulLoads ml;
  PS::mul_loads(ml, a, m, tc, col, step);
  cplx<T> v[R], w[R];
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = gload<T>(at_off(L, boff + unsigned(j) * jstride));
#pragma unroll
  for (int j = 0; j < R; ++j) w[j] = gload<T>(at_off(F, boff + unsigned(j) * jstride));
  const auto twsrc = [&]() {
    if constexpr (kWave) {
      TwRegs<T, N, R> r;
      load_twiddles<T, N, R>(r, tc, tw);
      return r;
    } else {
      return TwMem<T>{tw};
    }
  }();
  cplx<double> M[R];
  PS::multipliers(M, ml, a, m, tc, col, step, 1.0 / N);
  if constexpr (kWave) {
    const LdsRow<T> view_l{lds + cl * LSZ};
    team_fft_remap<T, N, R, -1>(v, tl, view_l, tc, view_c, twsrc);
    __syncthreads();  // the columns' arrays are free for the other transform's lanes
    team_fft_remap<T, N, R, -1>(w, tl, view_l, tc, view_c, twsrc);
  } else {
    team_fft<T, N, R, -1, View, Sync>(v, tc, view_c, twsrc);
    team_fft<T, N, R, -1, View, Sync>(w, tc, view_c, twsrc);
  }

  double acc[kAdjMom] = {0.0, 0.0, 0.0, 0.0};
  const double hd = a.hbar_half * m.dtheta;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const double u = hd * double(fidx(tc + j * TT, N)), u2 = u * u;
    // u^q Im(conj(v) w)
    double im = u * (double(v[j].x) * double(w[j].y) - double(v[j].y) * double(w[j].x));
#pragma unroll
    for (int q = 0; q < kAdjMom; ++q) {
      acc[q] += im;
      im *= u2;
    }
    v[j] = apply(v[j], cplx<double>{M[j].x, -M[j].y});  // conj(M_n) / P
  }
  if (m.theta_decay) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = apply(v[j], cplx<double>{gmem(m.theta_decay)[tc + j * TT], 0.0});
  }
  team_fft<T, N, R, +1, View, Sync>(v, tc, view_c, twsrc);
  if constexpr (kWave) {
    Sync::sync();
#pragma unroll
    for (int j = 0; j < R; ++j) *view_c.ptr(padr<R>(tc + j * TT)) = v[j];
    __syncthreads();
    const LdsRow<T> view_l{lds + cl * LSZ};
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = *view_l.ptr(padr<R>(tl + j * TT));
    // a column's lanes are TT consecutive lanes of one wave; the last one gets the sums
#pragma unroll
    for (int q = 0; q < kAdjMom; ++q) acc[q] = group_sum<TT>(acc[q]);
    if (tc == TT - 1) {
#pragma unroll
      for (int q = 0; q < kAdjMom; ++q) gmem(gcols)[size_t(col) * kAdjMom + q] = acc[q];
    }
  }
#pragma unroll
  for (int j = 0; j < R; ++j) store_cached(at_off(L, boff + unsigned(j) * jstride), v[j]);
  if constexpr (!kWave) {
    // lanes c + C*t of a wave hold column c: fold t, then across waves through LDS
#pragma unroll
    for (int off = C; off < 64; off <<= 1) {
#pragma unroll
      for (int q = 0; q < kAdjMom; ++q) acc[q] += __shfl_xor(acc[q], off, 64);
    }
    constexpr int kWaves = BLOCK / 64, kLanes = C < 64 ? C : 64;
    __syncthreads();
    double* red = reinterpret_cast<double*>(lds);
    const int wave = tid >> 6, lane = tid & 63;
    if (lane < kLanes) {
#pragma unroll
      for (int q = 0; q < kAdjMom; ++q) red[(wave * kLanes + lane) * kAdjMom + q] = acc[q];
    }
    __syncthreads();
    if (tid < C) {
#pragma unroll
      for (int q = 0; q < kAdjMom; ++q) {
        double s = 0.0;
        for (int k = 0; k < kWaves; ++k) s += red[(k * kLanes + tid) * kAdjMom + q];
        gmem(gcols)[size_t(tile * C + tid) * kAdjMom + q] = s;
      }
    }
  }
}

template <typename T, int R, int BLOCK>
__global__ void __launch_bounds__(BLOCK) adj_psweep_kernel(SweepArgs a, const void* W_next, double* gcols) {
  __shared__ cplx<T> lds[lds_elems<BLOCK, R>()];
  const unsigned w = p_item(a);
  CMember& m = member_at(a.members, 0);
  const int tile = int(w & 0xffffu);
  asm volatile("" ::"s"(m.X), "s"(m.P), "s"(m.pot), "s"(m.pot_deg), "s"(m.pot_rows), "s"(m.xmask),
               "s"(m.theta_decay), "s"(m.twP_hi), "s"(m.dx), "s"(m.dtheta));
#define BODY(n) adj_psweep_body<T, n, R, BLOCK>(a, m, tile, lds, W_next, gcols)
  WH_DISPATCH(m.P, BODY)
#undef BODY
}

// grad[s][k] = scale * sum_x g_k of the column moments of step s, one block per step:
// g_k = -2 sum_q C(k, q) x^(k-q) S_q.
__global__ void __launch_bounds__(256) grad_reduce_kernel(const Member* members, const double* gcols, double* grad,
                                                          double scale) {
  constexpr int K = kMaxDeg + 1, kWaves = 4;
  __shared__ double red[kWaves][K];
  CMember& m = member_at(members, 0);
  constexpr double binom[K][kAdjMom] = {{0, 0, 0, 0}, {1, 0, 0, 0},  {2, 0, 0, 0},   {3, 1, 0, 0},  {4, 4, 0, 0},
                                        {5, 10, 1, 0}, {6, 20, 6, 0}, {7, 35, 21, 1}, {8, 56, 56, 8}};
  const gptr<const double> cols = gmem(gcols) + size_t(blockIdx.x) * m.X * kAdjMom;
  double acc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0.0;
  for (int c = threadIdx.x; c < m.X; c += 256) {
    const double x = m.dx * double(fidx(c, m.X));
    double pw[K];
    pw[0] = 1.0;
#pragma unroll
    for (int k = 1; k < K; ++k) pw[k] = pw[k - 1] * x;
#pragma unroll
    for (int q = 0; q < kAdjMom; ++q) {
      const double s = -2.0 * cols[size_t(c) * kAdjMom + q];
#pragma unroll
      for (int k = 2 * q + 1; k < K; ++k) acc[k] += binom[k][q] * pw[k - 2 * q - 1] * s;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = group_sum<64>(acc[k]);
  if (lane == 63) {
#pragma unroll
    for (int k = 0; k < K; ++k) red[wave][k] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x < K) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += red[w][threadIdx.x];
    grad[size_t(blockIdx.x) * K + threadIdx.x] = scale * s;
  }
}

// Adjoint tile geometry: radix 8 (two register arrays per lane), 256 lanes a block, or 128 where those
// blocks would leave CUs idle (512^2: 11.3 -> 10.4 us a sweep).
constexpr int kAdjR = 8;
int adj_block(int X, int P) { return P <= 512 && X * P / (kAdjR * 256) < kCUs ? 128 : 256; }
int adj_cols(int X, int P) { return adj_block(X, P) / (P / kAdjR); }
size_t adj_moments(int X) { return size_t(X) * kAdjMom; }

template <typename T>
hipError_t adj_launch(int block, const SweepArgs& a, const void* W_next, double* gcols, hipStream_t s) {
  if (block == 128)
    hipLaunchKernelGGL((adj_psweep_kernel<T, kAdjR, 128>), dim3(a.ntiles), dim3(128), 0, s, a, W_next, gcols);
  else
    hipLaunchKernelGGL((adj_psweep_kernel<T, kAdjR, 256>), dim3(a.ntiles), dim3(256), 0, s, a, W_next, gcols);
  return hipGetLastError();
}
hipError_t launch_adj_psweep(int prec, int X, int P, const SweepArgs& a, const void* W_next, double* gcols,
                             hipStream_t s) {
  const int block = adj_block(X, P);
  return prec == 0 ? adj_launch<double>(block, a, W_next, gcols, s) : adj_launch<float>(block, a, W_next, gcols, s);
}

hipError_t launch_grad_reduce(const Member* members, const double* gcols, int nsteps, double* grad, double scale,
                              hipStream_t s) {
  hipLaunchKernelGGL(grad_reduce_kernel, dim3(nsteps), dim3(256), 0, s, members, gcols, grad, scale);
  return hipGetLastError();
}

}  // namespace wh
