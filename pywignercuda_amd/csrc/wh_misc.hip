// Reductions, small helpers and the plain axis transforms (cuFFT replacement).
//
//   colsum  column sums of a state (observables of a state not produced by a p sweep)
//   reduce  observables + complex norm of each member from its column sums,
//           renormalisation factor for the next load, Gross-Pitaevskii density
//           (GPU_Wigner2D_FFT.py:1778-1780, 1857-1878, 1912-1913; 435-455)
//   colpart_reduce  density after the kinetic step (GP.py:1933-1937)
//   fft_rows / fft_cols  in-place batched transforms for Plan_Z2Z_2D_Axis1 / Axis0
//           (cufft_wrapper.py:183-250, 396-403)
#include <hip/hip_runtime.h>

#include "wh_fft.hpp"
#include "wh_index.hpp"
#include "wh_kernels.hpp"

namespace wh {

// ------------------------------------------------------------------ column sums
// One tile = kColsumCols consecutive columns of one member; 256 lanes = 64 row groups of
// kColsumCols lanes (each load instruction of a wave covers 16 rows x 4 columns), the 64
// group sums combined by a fixed tree in LDS.
template <typename T>
__device__ __forceinline__ void colsum_tile(const Member& m, int tile, double (*red)[kColsumCols][kNCol]) {
  constexpr int CC = kColsumCols, G = 256 / CC;
  const cplx<T>* W = reinterpret_cast<const cplx<T>*>(m.W);
  const int c = threadIdx.x % CC, g = threadIdx.x / CC;
  const int col = tile * CC + c;
  double acc[kNCol] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (col < m.X) {
#pragma unroll 4
    for (int i = g; i < m.P; i += G) {
      const cplx<T> v = W[size_t(i) * m.X + col];
      const double p = m.p_host[i], wr = double(v.x);
      acc[0] += wr;
      acc[1] += double(v.y);
      acc[2] += p * wr;
      acc[3] += p * p * wr;
      acc[4] += wr < 0.0 ? wr : 0.0;
    }
  }
#pragma unroll
  for (int k = 0; k < kNCol; ++k) red[g][c][k] = acc[k];
  __syncthreads();
  for (int h = G / 2; h > 0; h >>= 1) {
    if (g < h) {
#pragma unroll
      for (int k = 0; k < kNCol; ++k) red[g][c][k] += red[g + h][c][k];
    }
    __syncthreads();
  }
  if (g == 0 && col < m.X) {
#pragma unroll
    for (int k = 0; k < kNCol; ++k) m.colsums[size_t(col) * kNCol + k] = red[0][c][k];
  }
}

template <typename T>
__global__ void __launch_bounds__(256) colsum_kernel(const Member* members, const unsigned* work) {
  __shared__ double red[256 / kColsumCols][kColsumCols][kNCol];
  const unsigned w = work[blockIdx.x];
  colsum_tile<T>(members[w >> 16], int(w & 0xffffu), red);
}

// ------------------------------------------------------------------ reduce (one block per member)
// One member's record row, pending factor and (Gross-Pitaevskii) density from its column
// sums, by a block of 256 threads.
__device__ __forceinline__ void reduce_member(const ReduceArgs& a, const Member& m, int step, double (*red)[256],
                                              double* scale_sh) {
  constexpr int K = 12;
  const int tid = threadIdx.x;
  double acc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0.0;
  for (int j = tid; j < m.X; j += 256) {
    const double* cs = m.colsums + size_t(j) * kNCol;
    const double s0 = cs[0], s0i = cs[1], s1 = cs[2], s2 = cs[3], sn = cs[4];
    const double x = m.x_host[j], dv = m.dv_host[j], v0 = m.v0_host[j];
    acc[0] += s0;
    acc[1] += s0i;
    acc[2] += x * s0;
    acc[3] += x * x * s0;
    acc[4] += s1;
    acc[5] += s2;
    acc[6] += x * s1;
    acc[7] += dv * s0;
    acc[8] += dv * s1;
    acc[9] += x * dv * s0;
    acc[10] += s2 * m.inv_2m + v0 * s0;
    acc[11] += sn;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) red[k][tid] = acc[k];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (tid < h) {
#pragma unroll
      for (int k = 0; k < K; ++k) red[k][tid] += red[k][tid + h];
    }
    __syncthreads();
  }
  if (tid == 0) {
    // W_normalised = W / n, n = dXdP sum W (complex); observables are Re(dXdP sum W A / n)
    // = dXdP Re(sum W A) nr / |n|^2 up to Im(sum W A) ni / |n|^2 (below 1e-30 here)
    const double nr = m.dxdp * red[0][0], ni = m.dxdp * red[1][0];
    double f = 1.0, sr = 1.0, si = 0.0;
    if (a.renorm) {
      const double m2 = nr * nr + ni * ni;
      f = nr / m2;
      sr = nr / m2;
      si = -ni / m2;
    }
    scale_sh[0] = sr;
    scale_sh[1] = si;
    if (a.update_scale) {
      m.scale[0] = sr;
      m.scale[1] = si;
    }
    if (a.record) {
      double* o = m.obs + size_t(step - m.obs_base) * kNObs;
      const double d = m.dxdp * f;
      o[kObsX] = d * red[2][0];
      o[kObsX2] = d * red[3][0];
      o[kObsP] = d * red[4][0];
      o[kObsP2] = d * red[5][0];
      o[kObsXP] = d * red[6][0];
      o[kObsDV] = d * red[7][0];
      o[kObsPDV] = d * red[8][0];
      o[kObsXDV] = d * red[9][0];
      o[kObsH] = d * red[10][0];
      o[kObsNeg] = d * red[11][0];
      o[kObsNorm] = d * red[0][0];
      o[kObsRawNormRe] = nr;
      o[kObsRawNormIm] = ni;
    }
  }
  if (a.rho) {
    __syncthreads();
    const double sr = scale_sh[0], si = scale_sh[1];
    for (int j = tid; j < m.X; j += 256) {
      const double* cs = m.colsums + size_t(j) * kNCol;
      m.rho[j] = (cs[0] * sr - cs[1] * si) * m.rho_factor;
    }
  }
}

// ------------------------------------------------------------------ reduce (one block per member)
__global__ void __launch_bounds__(256) reduce_kernel(ReduceArgs a, int* done, int nblocks) {
  __shared__ double red[12][256];
  __shared__ double scale_sh[2];
  const int step = a.use_step_arg ? a.step_arg : *a.step;
  reduce_member(a, a.members[blockIdx.x], step, red, scale_sh);
  if (a.step_inc && threadIdx.x == 0) {
    // the last block to finish advances the step counter: every block has read it by then
    __threadfence();
    const int prev = atomicAdd(done, 1);
    if (prev == nblocks - 1) {
      *done = 0;
      *a.step_inc = a.next_step >= 0 ? a.next_step : step + 1;
      __threadfence();
    }
  }
}

// ------------------------------------------------------------------ density after K
// rho(x) from the x sweep's partial sums [tiles][X].  One work item = COLS columns of one
// member, 256 / COLS groups of lanes each summing every (256 / COLS)-th tile.  (One block
// per member, a column per lane and all tiles in its loop, took 28 us at 512^2.)
template <int COLS>
__global__ void __launch_bounds__(256) colpart_reduce_kernel(const Member* members, int xradix, int xblock) {
  constexpr int G = 256 / COLS;
  __shared__ double red[G][COLS];
  CMember& m = member_at(members, blockIdx.y);
  const int nblk = m.P / (xblock / (m.X / xradix));  // x-sweep tiles of this member
  const int c = threadIdx.x % COLS, g = threadIdx.x / COLS;
  const int x = blockIdx.x * COLS + c;
  if (int(blockIdx.x) * COLS >= m.X) return;  // the grid spans the widest member (X is a multiple of COLS)
  const gptr<const double> part = gmem(const_cast<const double*>(m.colpart));
  double s = 0.0;
#pragma unroll 8
  for (int b = g; b < nblk; b += G) s += part[size_t(b) * m.X + x];
  red[g][c] = s;
  __syncthreads();
  if (g == 0) {
    s = 0.0;
#pragma unroll
    for (int k = 0; k < G; ++k) s += red[k][c];
    gmem(m.rho)[x] = s * m.rho_factor;
  }
}

// ------------------------------------------------------------------ scale by the pending factor
template <typename T>
__global__ void __launch_bounds__(256) scale_kernel(const Member* members, const unsigned* work) {
  const unsigned w = work[blockIdx.x];
  const Member& m = members[w >> 16];
  const size_t chunk = size_t(w & 0xffffu) * kScaleChunk;
  const size_t n = size_t(m.X) * size_t(m.P);
  cplx<T>* W = reinterpret_cast<cplx<T>*>(m.W);
  // all of this thread's loads in flight before the factor arrives and the stores start
  static_assert(kScaleChunk % 256 == 0, "whole elements per thread");
  constexpr int kPer = kScaleChunk / 256;
  cplx<T> v[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const size_t i = chunk + threadIdx.x + size_t(k) * 256;
    if (i < n) v[k] = W[i];
  }
  const double sr = m.scale[0], si = m.scale[1];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const size_t i = chunk + threadIdx.x + size_t(k) * 256;
    if (i < n) {
      const double x = double(v[k].x), y = double(v[k].y);
      W[i] = {T(x * sr - y * si), T(x * si + y * sr)};
    }
  }
}

__global__ void set_int_kernel(int* p, int v) { *p = v; }
__global__ void bind_kernel(BindArgs a) {
  const int i = threadIdx.x;
  if (i < a.count) {
    Member& m = a.members[a.first + i];
    m.W = a.W[i];
    m.obs = a.obs[i];
    m.obs_base = a.obs_base;
  }
}
__global__ void set_scale_kernel(const Member* members, double re, double im) {
  const Member& m = members[blockIdx.x];
  if (threadIdx.x == 0) {
    m.scale[0] = re;
    m.scale[1] = im;
  }
}

// ------------------------------------------------------------------ plain axis transforms
// Teams of one wave (radix 8 up to N = 512, radix 16 at 1024) exchange without block barriers and hold
// their twiddles in registers, loaded with the state.  A row block is one wave (or the team), so that
// a few hundred rows reach every CU: blocks of 256 lanes left half of them idle at 512 x 1024.
// A forward and an inverse pair over both axes with two clones, us, before -> after (radix 16 for every
// length, block barriers, 256 lanes a block): 2048^2 complex128 239 -> 147, complex64 205 -> 119; 1024^2
// 65 -> 60 and 64 -> 44; 512 x 1024 47 -> 38; below, the calls' host time (38 us) covers the kernels.
template <typename T, int N>
struct FftShape {
  static constexpr int R = N <= 512 ? 8 : 16, TT = N / R;
  static constexpr bool kWave = TT <= 64;
  static constexpr int ROWS = TT >= 64 ? 1 : 64 / TT;             // rows per block
  static constexpr int C = N <= 64 ? 8 : N <= 1024 ? 4 : 2;      // columns per block
  using Sync = std::conditional_t<kWave, WaveSync, BlockSync>;
};

template <typename T, int N, int DIR>
__global__ void __launch_bounds__((FftShape<T, N>::ROWS * FftShape<T, N>::TT))
    fft_rows_kernel(void* data, int rows, int normalize, Twiddles<T> tw) {
  using G = FftShape<T, N>;
  constexpr int R = G::R, TT = G::TT, ROWS = G::ROWS;
  constexpr int LSZ = Padded<N, R>::size;
  __shared__ cplx<T> lds[ROWS * LSZ];
  const int tid = threadIdx.x;
  const int team = tid / TT, t = tid % TT;
  const int row = blockIdx.x * ROWS + team;
  const bool active = row < rows;
  const gptr<cplx<T>> W = gmem(reinterpret_cast<cplx<T>*>(data)) + size_t(active ? row : 0) * N;
  LdsRow<T> view{lds + team * LSZ};
  TwRegs<T, N, R> twr;
  load_twiddles<T, N, R>(twr, t, tw);
  cplx<T> v[R];
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = gload(W + t + j * TT);
  team_fft<T, N, R, DIR, LdsRow<T>, typename G::Sync>(v, t, view, twr);
  const T f = normalize ? T(1.0 / N) : T(1);
  if (active) {
#pragma unroll
    for (int j = 0; j < R; ++j) store_cached(W + t + j * TT, cscale(v[j], f));
  }
}

// Loads and stores cover rows of C consecutive columns; a wave's team takes its column over at the
// first exchange and hands it back before the store.
template <typename T, int N, int DIR>
__global__ void __launch_bounds__((FftShape<T, N>::C * FftShape<T, N>::TT))
    fft_cols_kernel(void* data, int X, int normalize, Twiddles<T> tw) {
  using G = FftShape<T, N>;
  constexpr int R = G::R, TT = G::TT, C = G::C;
  constexpr int LSZ = N + N / R + col_pad<T, C>();
  __shared__ cplx<T> lds[C * LSZ];
  const int tid = threadIdx.x;
  const int cl = tid % C, tl = tid / C;
  const int cc = G::kWave ? tid / TT : cl, tc = G::kWave ? tid % TT : tl;
  // neighbouring tiles, which share 128-byte lines, on one XCD
  const int nt = int(gridDim.x), b = int(blockIdx.x);
  const int tile = nt % 8 == 0 ? (b % 8) * (nt / 8) + b / 8 : b;
  const gptr<cplx<T>> W = gmem(reinterpret_cast<cplx<T>*>(data)) + col_element(tl, X, tile * C + cl);
  TwRegs<T, N, R> twr;
  load_twiddles<T, N, R>(twr, tc, tw);
  cplx<T> v[R];
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = gload(W + col_element(j * TT, X, 0));
  if constexpr (G::kWave) {
    const LdsRow<T> view_l{lds + cl * LSZ}, view_c{lds + cc * LSZ};
    team_fft_remap<T, N, R, DIR>(v, tl, view_l, tc, view_c, twr);
    WaveSync::sync();
#pragma unroll
    for (int j = 0; j < R; ++j) *view_c.ptr(padr<R>(tc + j * TT)) = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = *view_l.ptr(padr<R>(tl + j * TT));
  } else {
    team_fft<T, N, R, DIR, LdsStrided<T, C>, BlockSync>(v, tl, LdsStrided<T, C>{lds + cl}, twr);
  }
  const T f = normalize ? T(1.0 / N) : T(1);
#pragma unroll
  for (int j = 0; j < R; ++j) store_cached(W + col_element(j * TT, X, 0), cscale(v[j], f));
}

// ------------------------------------------------------------------ launchers
namespace {
constexpr int kR = 16;
// columns a plan's batch has to be a multiple of (a multiple of every kernel's C)
template <typename T, int N>
constexpr int fft_cols_per_block() {
  constexpr int c = 256 / (N / kR);
  static_assert((c > 64 ? 64 : c) % FftShape<T, N>::C == 0, "whole tiles");
  return c < 1 ? 1 : (c > 64 ? 64 : c);
}
template <typename T, int N, int DIR>
hipError_t fft_rows_n(void* d, int rows, int norm, Twiddles<T> tw, hipStream_t s) {
  using G = FftShape<T, N>;
  hipLaunchKernelGGL((fft_rows_kernel<T, N, DIR>), dim3((rows + G::ROWS - 1) / G::ROWS), dim3(G::ROWS * G::TT), 0, s,
                     d, rows, norm, tw);
  return hipGetLastError();
}
template <typename T, int N, int DIR>
hipError_t fft_cols_n(void* d, int X, int norm, Twiddles<T> tw, hipStream_t s) {
  using G = FftShape<T, N>;
  hipLaunchKernelGGL((fft_cols_kernel<T, N, DIR>), dim3(X / G::C), dim3(G::C * G::TT), 0, s, d, X, norm, tw);
  return hipGetLastError();
}
#define WH_FFT_SWITCH(N, CALL)         \
  switch (N) {                         \
    case 64: return CALL(64);          \
    case 128: return CALL(128);        \
    case 256: return CALL(256);        \
    case 512: return CALL(512);        \
    case 1024: return CALL(1024);      \
    case 2048: return CALL(2048);      \
    default: return hipErrorInvalidValue; \
  }
template <typename T, int DIR>
hipError_t rows_t(int N, void* d, int rows, int norm, Twiddles<T> tw, hipStream_t s) {
#define CALL(n) fft_rows_n<T, n, DIR>(d, rows, norm, tw, s)
  WH_FFT_SWITCH(N, CALL)
#undef CALL
}
template <typename T, int DIR>
hipError_t cols_t(int N, void* d, int X, int norm, Twiddles<T> tw, hipStream_t s) {
#define CALL(n) fft_cols_n<T, n, DIR>(d, X, norm, tw, s)
  WH_FFT_SWITCH(N, CALL)
#undef CALL
}
}  // namespace

int fft_cols_batch_multiple(int prec, int N) {
  switch (N) {
    case 64: return prec == 0 ? fft_cols_per_block<double, 64>() : fft_cols_per_block<float, 64>();
    case 128: return prec == 0 ? fft_cols_per_block<double, 128>() : fft_cols_per_block<float, 128>();
    case 256: return prec == 0 ? fft_cols_per_block<double, 256>() : fft_cols_per_block<float, 256>();
    case 512: return prec == 0 ? fft_cols_per_block<double, 512>() : fft_cols_per_block<float, 512>();
    case 1024: return prec == 0 ? fft_cols_per_block<double, 1024>() : fft_cols_per_block<float, 1024>();
    case 2048: return prec == 0 ? fft_cols_per_block<double, 2048>() : fft_cols_per_block<float, 2048>();
    default: return 0;
  }
}

hipError_t launch_fft_axis(int prec, int columns, int N, int dir, void* d, int batch, int norm,
                           const void* tw_hi, const void* tw_lo, hipStream_t s) {
  if (prec == 0) {
    Twiddles<double> tw{static_cast<const cplx<double>*>(tw_hi), nullptr};
    if (columns) return dir < 0 ? cols_t<double, -1>(N, d, batch, norm, tw, s) : cols_t<double, 1>(N, d, batch, norm, tw, s);
    return dir < 0 ? rows_t<double, -1>(N, d, batch, norm, tw, s) : rows_t<double, 1>(N, d, batch, norm, tw, s);
  }
  Twiddles<float> tw{static_cast<const cplx<float>*>(tw_hi), static_cast<const cplx<float>*>(tw_lo)};
  if (columns) return dir < 0 ? cols_t<float, -1>(N, d, batch, norm, tw, s) : cols_t<float, 1>(N, d, batch, norm, tw, s);
  return dir < 0 ? rows_t<float, -1>(N, d, batch, norm, tw, s) : rows_t<float, 1>(N, d, batch, norm, tw, s);
}

hipError_t launch_colsum(int prec, const Member* members, const unsigned* work, int nwork, hipStream_t s) {
  if (prec == 0)
    hipLaunchKernelGGL(colsum_kernel<double>, dim3(nwork), dim3(256), 0, s, members, work);
  else
    hipLaunchKernelGGL(colsum_kernel<float>, dim3(nwork), dim3(256), 0, s, members, work);
  return hipGetLastError();
}
hipError_t launch_reduce(const ReduceArgs& a, int nmembers, int* done, hipStream_t s) {
  hipLaunchKernelGGL(reduce_kernel, dim3(nmembers), dim3(256), 0, s, a, done, nmembers);
  return hipGetLastError();
}
hipError_t launch_colpart_reduce(const Member* members, int nmembers, int max_x, int xradix, int xblock,
                                 hipStream_t s) {
  // 16 columns (one 128-byte line per row of partials) and 16 lane groups
  constexpr int COLS = 16;
  hipLaunchKernelGGL(colpart_reduce_kernel<COLS>, dim3(max_x / COLS, nmembers), dim3(256), 0, s, members, xradix,
                     xblock);
  return hipGetLastError();
}
hipError_t launch_scale(int prec, const Member* members, const unsigned* work, int nwork, hipStream_t s) {
  if (prec == 0)
    hipLaunchKernelGGL(scale_kernel<double>, dim3(nwork), dim3(256), 0, s, members, work);
  else
    hipLaunchKernelGGL(scale_kernel<float>, dim3(nwork), dim3(256), 0, s, members, work);
  return hipGetLastError();
}
hipError_t launch_set_int(int* p, int v, hipStream_t s) {
  hipLaunchKernelGGL(set_int_kernel, dim3(1), dim3(1), 0, s, p, v);
  return hipGetLastError();
}
hipError_t launch_bind(const BindArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(bind_kernel, dim3(1), dim3(64), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_set_scale(const Member* members, int nmembers, double re, double im, hipStream_t s) {
  hipLaunchKernelGGL(set_scale_kernel, dim3(nmembers), dim3(64), 0, s, members, re, im);
  return hipGetLastError();
}

}  // namespace wh
