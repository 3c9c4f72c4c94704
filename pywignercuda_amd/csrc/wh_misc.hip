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
#include "wh_variants.hpp"

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
// Narrow form: teams of one wave (radix 8 up to N = 512, radix 16 at 1024) exchange without block barriers
// and hold their twiddles in registers, loaded with the state.  A row block is one wave (or the team), so
// that a few hundred rows reach every CU: blocks of 256 lanes left half of them idle at 512 x 1024.
// A forward and an inverse pair over both axes with two clones, us, against radix 16, block barriers and
// 256 lanes a block for every length: 2048^2 complex128 239 -> 147, complex64 205 -> 119; 1024^2
// 65 -> 60 and 64 -> 44; 512 x 1024 47 -> 38; below, the calls' host time (38 us) covers the kernels.
// Complex128 radix-8 teams carry sqrt(1/2) with its low part (ConstMul): <q^2> of a Gaussian after 72
// forward and inverse transforms of 128..512 is 6e-16 to 4e-15 off, without it 8e-14 to 1.3e-13, with
// radix 16 6e-15 to 1.7e-14; at most 0.2 us a call.
// Wide form (large batches, the rules are in fft_rows_n and fft_cols_n): radix 16 in blocks of 256 lanes.
// Its rows of columns are whole 128-byte lines (64 bytes at complex64 512) and it exchanges once less; a
// narrow block's rows of 4 columns are 32 or 64 bytes, too short once the batch is beyond the L2s.
template <typename T, int N, bool WIDE>
struct FftShape {
  static constexpr int R = WIDE || N > 512 ? 16 : 8, TT = N / R;
  static constexpr int kLines = 256 / TT < 1 ? 1 : 256 / TT;                                // of a wide block
  static constexpr int ROWS = WIDE ? kLines : TT >= 64 ? 1 : 64 / TT;                       // rows per block
  static constexpr int C = WIDE ? (kLines > 64 ? 64 : kLines) : N <= 64 ? 8 : N <= 1024 ? 4 : 2;  // columns per block
  // teams of one wave; wide rows only in FP32, where they are faster (512 x 32768: 43 us, with block
  // barriers 47; FP64 the other way round beyond the caches: 512 x 262144 727 and 805)
  static constexpr bool kWaveRows = TT <= 64 && (!WIDE || sizeof(T) == 4), kWaveCols = TT <= 64 && !WIDE;
};

template <bool REGS, typename T, int N, int R>
__device__ __forceinline__ auto fft_twiddles(int t, const Twiddles<T>& tw) {
  if constexpr (REGS) {
    TwRegs<T, N, R, sizeof(T) == 8 && R == 8> r;
    load_twiddles<T, N, R>(r, t, tw);
    return r;
  } else {
    return TwMem<T>{tw};
  }
}

template <typename T, int N, bool WIDE, int DIR>
__global__ void __launch_bounds__((FftShape<T, N, WIDE>::ROWS * FftShape<T, N, WIDE>::TT))
    fft_rows_kernel(void* data, int rows, int normalize, Twiddles<T> tw) {
  using G = FftShape<T, N, WIDE>;
  using Sync = std::conditional_t<G::kWaveRows, WaveSync, BlockSync>;
  constexpr int R = G::R, TT = G::TT, ROWS = G::ROWS;
  constexpr int LSZ = Padded<N, R>::size;
  __shared__ cplx<T> lds[ROWS * LSZ];
  const int tid = threadIdx.x;
  const int team = tid / TT, t = tid % TT;
  const int row = blockIdx.x * ROWS + team;
  const bool active = row < rows;
  const gptr<cplx<T>> W = gmem(reinterpret_cast<cplx<T>*>(data)) + size_t(active ? row : 0) * N;
  LdsRow<T> view{lds + team * LSZ};
  const auto twsrc = fft_twiddles<!WIDE, T, N, R>(t, tw);
  cplx<T> v[R];
  if constexpr (G::kWaveRows || !WIDE) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = gload(W + t + j * TT);
  } else {
    // in a branch, in front of which the compiler moves no twiddle load (2048 x 65536 complex128:
    // 728 us, without the branch 764)
#pragma unroll
    for (int j = 0; j < R; ++j) {
      v[j] = {T(0), T(0)};
      if (active) v[j] = gload(W + t + j * TT);
    }
  }
  team_fft<T, N, R, DIR, LdsRow<T>, Sync>(v, t, view, twsrc);
  const T f = normalize ? T(1.0 / N) : T(1);
  if (active) {
#pragma unroll
    for (int j = 0; j < R; ++j) store_cached(W + t + j * TT, cscale(v[j], f));
  }
}

// Loads and stores cover rows of C consecutive columns; a wave's team takes its column over at the
// first exchange and hands it back before the store.  FAR: offsets in 64 bits (offsets_fit_32).
template <typename T, int N, bool WIDE, bool FAR, int DIR>
__global__ void __launch_bounds__((FftShape<T, N, WIDE>::C * FftShape<T, N, WIDE>::TT))
    fft_cols_kernel(void* data, int X, int normalize, Twiddles<T> tw) {
  using G = FftShape<T, N, WIDE>;
  constexpr int R = G::R, TT = G::TT, C = G::C;
  constexpr int LSZ = G::kWaveCols ? N + N / R + col_pad<T, C>() : Padded<N, R>::size;
  __shared__ cplx<T> lds[C * LSZ];
  const int tid = threadIdx.x;
  const int cl = tid % C, tl = tid / C;
  const int cc = G::kWaveCols ? tid / TT : cl, tc = G::kWaveCols ? tid % TT : tl;
  // neighbouring tiles that share 128-byte lines on one XCD (whole lines go in order: complex128
  // 256 x 131072 204 us, by XCD 217)
  constexpr bool kShared = C * int(sizeof(cplx<T>)) < 128;
  const int nt = int(gridDim.x), b = int(blockIdx.x);
  const int tile = kShared && nt % 8 == 0 ? (b % 8) * (nt / 8) + b / 8 : b;
  const gptr<cplx<T>> W = gmem(reinterpret_cast<cplx<T>*>(data));
  const int col = tile * C + cl;
  const unsigned boff = (unsigned(tl) * unsigned(X) + unsigned(col)) * unsigned(sizeof(cplx<T>));
  const auto element = [&](int j) {
    if constexpr (FAR)
      return W + col_element(tl + j * TT, X, col);
    else
      return at_off(W + col_element(j * TT, X, 0), boff);
  };
  const auto twsrc = fft_twiddles<!WIDE, T, N, R>(tc, tw);
  cplx<T> v[R];
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = gload(element(j));
  if constexpr (G::kWaveCols) {
    const LdsRow<T> view_l{lds + cl * LSZ}, view_c{lds + cc * LSZ};
    team_fft_remap<T, N, R, DIR>(v, tl, view_l, tc, view_c, twsrc);
    WaveSync::sync();
#pragma unroll
    for (int j = 0; j < R; ++j) *view_c.ptr(padr<R>(tc + j * TT)) = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = *view_l.ptr(padr<R>(tl + j * TT));
  } else {
    team_fft<T, N, R, DIR, LdsStrided<T, C>, BlockSync>(v, tl, LdsStrided<T, C>{lds + cl}, twsrc);
  }
  const T f = normalize ? T(1.0 / N) : T(1);
#pragma unroll
  for (int j = 0; j < R; ++j) store_cached(element(j), cscale(v[j], f));
}

// ------------------------------------------------------------------ launchers
namespace {
constexpr int kR = 16;
constexpr size_t kLargeBatch = size_t(512) << 20;  // bytes: twice the last-level cache
// columns a plan's batch has to be a multiple of (a multiple of every kernel's C)
template <typename T, int N>
constexpr int fft_cols_per_block() {
  constexpr int c = 256 / (N / kR), cols = c < 1 ? 1 : (c > 64 ? 64 : c);
  static_assert(cols % FftShape<T, N, false>::C == 0 && cols % FftShape<T, N, true>::C == 0, "whole tiles");
  return cols;
}
template <typename T, int N, bool WIDE, int DIR>
hipError_t fft_rows_form(void* d, int rows, int norm, Twiddles<T> tw, hipStream_t s) {
  using G = FftShape<T, N, WIDE>;
  hipLaunchKernelGGL((fft_rows_kernel<T, N, WIDE, DIR>), dim3((rows + G::ROWS - 1) / G::ROWS), dim3(G::ROWS * G::TT), 0,
                     s, d, rows, norm, tw);
  return hipGetLastError();
}
// Wide rows: complex64 of 128..512 from a wide block per CU on (us, narrow -> wide: 512 x 4096 11.1 -> 8.6,
// 512 x 32768 64.3 -> 43.2, 256 x 32768 24.8 -> 22.5, 128 x 32768 11.5 -> 9.7), every type and length
// from 512 MiB on, twice the last-level cache (complex128 2048 x 65536 807 -> 728, 512 x 262144 767 -> 727,
// 256 x 262144 398 -> 373; below that the narrow form: 512 x 32768 63.0 and 71.2).
template <typename T, int N, int DIR>
hipError_t fft_rows_n(void* d, int rows, int norm, Twiddles<T> tw, hipStream_t s) {
  const bool many = sizeof(T) == 4 && N >= 128 && N <= 512 && rows / FftShape<T, N, true>::ROWS >= kCUs;
  const bool large = size_t(rows) * N * sizeof(cplx<T>) >= kLargeBatch;
  return many || large ? fft_rows_form<T, N, true, DIR>(d, rows, norm, tw, s)
                       : fft_rows_form<T, N, false, DIR>(d, rows, norm, tw, s);
}
template <typename T, int N, bool WIDE, bool FAR, int DIR>
hipError_t fft_cols_form(void* d, int X, int norm, Twiddles<T> tw, hipStream_t s) {
  using G = FftShape<T, N, WIDE>;
  hipLaunchKernelGGL((fft_cols_kernel<T, N, WIDE, FAR, DIR>), dim3(X / G::C), dim3(G::C * G::TT), 0, s, d, X, norm, tw);
  return hipGetLastError();
}
// Wide columns up to N = 512 from a wide block per CU on (us, narrow -> wide: complex64 128 x 32768
// 15.2 -> 10.2, 256 x 8192 10.5 -> 7.6, 512 x 4096 13.4 -> 8.0; complex128 512 x 4096 12.3 -> 10.1,
// 256 x 262144 579 -> 414; below that 256 x 2048 4.9 -> 5.1).  Complex128 of 64, whose narrow rows of 8
// columns are whole lines, only from 512 MiB on (64 x 32768 8.1 -> 10.9, 64 x 524288 225 -> 196).  At 1024
// and 2048 a narrow block has as many columns.
template <typename T, int N, int DIR>
hipError_t fft_cols_n(void* d, int X, int norm, Twiddles<T> tw, hipStream_t s) {
  if (!offsets_fit_32(FftShape<T, N, (N <= 512)>::TT, X, sizeof(cplx<T>)))  // 64 GiB and more
    return fft_cols_form<T, N, (N <= 512), true, DIR>(d, X, norm, tw, s);
  if constexpr (N <= 512) {
    const bool many = (sizeof(T) == 4 || N >= 128) && X / FftShape<T, N, true>::C >= kCUs;
    const bool large = size_t(X) * N * sizeof(cplx<T>) >= kLargeBatch;
    if (many || large) return fft_cols_form<T, N, true, false, DIR>(d, X, norm, tw, s);
  }
  return fft_cols_form<T, N, false, false, DIR>(d, X, norm, tw, s);
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
hipError_t launch_bind(const BindArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(bind_kernel, dim3(1), dim3(64), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_set_scale(const Member* members, int nmembers, double re, double im, hipStream_t s) {
  hipLaunchKernelGGL(set_scale_kernel, dim3(nmembers), dim3(64), 0, s, members, re, im);
  return hipGetLastError();
}

}  // namespace wh
