// Device-side FFT building blocks for gfx950 (CDNA4), wave64.
//
// A "team" of TT = N/R lanes computes one length-N complex transform.  Lane t
// holds R elements in registers in the strided layout  v[j] = a[t + j*TT].
// The transform is a Stockham autosort sequence of radix passes [R, R, ..., r]
// (r = N / R^k).  The first pass works on the registers directly, every later
// pass exchanges through LDS, and the last pass writes back into the same
// strided register layout.  So a forward transform, a pointwise multiply and an
// inverse transform chain in registers, and global loads and stores of the
// strided layout are coalesced for row teams and column teams alike.
//
// Pass with radix r after the span Ns = prod(previous radices):
//   butterfly b in [0, N/r) reads a[b + j*N/r], twiddles by w^(j*(b mod Ns)),
//   w = exp(dir*2*pi*i/(Ns*r)), applies an r-point DFT and writes
//   a'[(b - b mod Ns)*r + (b mod Ns) + q*Ns].
// Twiddles come from a table tw[n] = exp(-2*pi*i*n/N) computed in FP64 on the
// host.  Forward = exponent -i (dir = -1), inverse = +i and unnormalised, as
// cufftExecZ2Z (cufft_wrapper.py:11-12, 81-103).
//
// FP32: every constant the transform multiplies by (table twiddles and the
// in-register radix-16 roots) is carried as a hi + lo float pair, so the
// transform's operator is exact to ~2^-48 and only value-dependent rounding
// remains: a fixed perturbation of the step operator would accumulate linearly
// over thousands of unitary steps, rounding noise only as a random walk.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace wh {

template <typename T>
struct alignas(2 * sizeof(T)) cplx {
  T x, y;
};

// Address-space qualified pointers.  Pointers that reach device code through memory
// (tables, member records) are generic, for which the compiler emits flat_ instructions;
// those also count against the LDS counter, so every LDS wait of an exchange would
// wait for outstanding memory loads as well.  gptr: global memory (global_ loads and
// stores).  cptr: read-only for the whole kernel (uniform addresses load through the
// scalar cache; never written through).
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
using cptr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> gmem(T* p) {
  return (gptr<T>)p;
}
template <typename T>
__device__ __forceinline__ cptr<T> cmem(const T* p) {
  return (cptr<T>)p;
}
// complex element through a global pointer (one 2-vector load)
template <typename T>
__device__ __forceinline__ cplx<T> gload(gptr<const cplx<T>> p) {
  typedef T vec2 __attribute__((ext_vector_type(2)));
  const vec2 r = *reinterpret_cast<gptr<const vec2>>(p);
  return {r.x, r.y};
}
template <typename T>
__device__ __forceinline__ cplx<T> gload(gptr<cplx<T>> p) {
  return gload<T>(gptr<const cplx<T>>(p));
}

// element of a uniform row base at a per-lane 32-bit byte offset (SGPR base +
// VGPR offset addressing: one offset register per lane for all strided elements)
template <typename T>
__device__ __forceinline__ cplx<T>& at_off(cplx<T>* base, unsigned boff) {
  return *reinterpret_cast<cplx<T>*>(reinterpret_cast<char*>(base) + boff);
}
template <typename T>
__device__ __forceinline__ gptr<cplx<T>> at_off(gptr<cplx<T>> base, unsigned boff) {
  return reinterpret_cast<gptr<cplx<T>>>(reinterpret_cast<gptr<char>>(base) + boff);
}
template <typename T>
__device__ __forceinline__ gptr<const cplx<T>> at_off(gptr<const cplx<T>> base, unsigned boff) {
  return reinterpret_cast<gptr<const cplx<T>>>(reinterpret_cast<gptr<const char>>(base) + boff);
}

// Streaming store of a state element: the sweep writes each element once and the next
// sweep reads it from another CU, so the line is not kept dirty in this CU's L2 (less
// write-back at the end of the kernel).
template <typename S>
__device__ __forceinline__ void store_stream(gptr<cplx<S>> p, cplx<S> v) {
  typedef S vec2 __attribute__((ext_vector_type(2)));
  __builtin_nontemporal_store(vec2{v.x, v.y}, reinterpret_cast<gptr<vec2>>(p));
}

// Write-back store of a state element, for sweeps whose store instruction covers half of
// each 128-byte line (the p sweep's C-column rows): the neighbouring tile, on the same XCD at
// about the same time, fills the other half in L2 before the line is written back.  With
// streaming stores the half lines went out separately (+39% WRITE_SIZE on a 64 x 1024^2
// FP64 batch; +1.2% with this store).
template <typename S>
__device__ __forceinline__ void store_cached(gptr<cplx<S>> p, cplx<S> v) {
  typedef S vec2 __attribute__((ext_vector_type(2)));
  *reinterpret_cast<gptr<vec2>>(p) = vec2{v.x, v.y};
}

template <typename T>
__device__ __forceinline__ cplx<T> cadd(cplx<T> a, cplx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ cplx<T> csub(cplx<T> a, cplx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ __forceinline__ cplx<T> cscale(cplx<T> a, T s) { return {a.x * s, a.y * s}; }

constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n / 2); }
constexpr int ipow(int b, int e) { return e == 0 ? 1 : b * ipow(b, e - 1); }
// number of Stockham passes for N with maximal radix R
constexpr int num_passes(int N, int R) { return N <= R ? 1 : 1 + num_passes(N / R, R); }
// radix of pass p (all R except possibly the last)
constexpr int pass_radix(int N, int R, int p) {
  return (p == num_passes(N, R) - 1) ? N / ipow(R, p) : R;
}
constexpr int bitrev(int v, int bits) {
  return bits == 0 ? 0 : ((v & 1) << (bits - 1)) | bitrev(v >> 1, bits - 1);
}

// cos(2*pi*k/16), k = 0..15
constexpr double cos16(int k) {
  constexpr double c1 = 0.92387953251128675613;  // cos(pi/8)
  constexpr double c2 = 0.70710678118654752440;  // cos(pi/4)
  constexpr double c3 = 0.38268343236508977173;  // cos(3pi/8)
  const double t[16] = {1.0, c1, c2, c3, 0.0, -c3, -c2, -c1, -1.0, -c1, -c2, -c3, 0.0, c3, c2, c1};
  return t[k & 15];
}

constexpr double kHalfRootLow = -4.8336466567264565186e-17;  // sqrt(1/2) less the double next to it

// a * (c + i s) with constants known at compile time; FP32 adds the products
// with the low parts of the constants.
// EXACT (FP64, odd multiples of pi/4): with the low part of sqrt(1/2).  Its rounding scales half of a
// radix-8 butterfly's terms by 1 - 7e-17 in every pass and both directions, a fixed perturbation that
// adds up over the steps: <p^2> after 72 steps at P = 1024 is 8.7e-13 off with it (radix 16: 1.7e-13).
template <typename T>
struct ConstMul;
template <>
struct ConstMul<double> {
  template <int K, int DIR, bool EXACT>
  __device__ __forceinline__ static cplx<double> mul(cplx<double> a) {
    constexpr double C = cos16(K), S = (DIR < 0 ? -1.0 : 1.0) * cos16(K + 12);
    if constexpr (EXACT && K % 4 == 2) {  // C (1 +- i), the low part added before the one rounding
      constexpr double lo = C > 0.0 ? kHalfRootLow : -kHalfRootLow;
      const double d = (S > 0.0) == (C > 0.0) ? a.x - a.y : a.x + a.y;
      const double e = (S > 0.0) == (C > 0.0) ? a.x + a.y : a.y - a.x;
      return {fma(d, C, d * lo), fma(e, C, e * lo)};
    }
    return {a.x * C - a.y * S, a.x * S + a.y * C};
  }
};
template <>
struct ConstMul<float> {
  template <int K, int DIR, bool EXACT>
  __device__ __forceinline__ static cplx<float> mul(cplx<float> a) {
    constexpr double C = cos16(K), S = (DIR < 0 ? -1.0 : 1.0) * cos16(K + 12);
    constexpr float ch = float(C), sh = float(S);
    constexpr float cl = float(C - double(ch)), sl = float(S - double(sh));
    const float rx = fmaf(a.x, ch, -a.y * sh), ry = fmaf(a.x, sh, a.y * ch);
    return {rx + fmaf(a.x, cl, -a.y * sl), ry + fmaf(a.x, sl, a.y * cl)};
  }
};

// a * exp(DIR * 2*pi*i * K / M), M | 16; the special angles are exact.
template <int DIR, int K, int M, bool EXACT, typename T>
__device__ __forceinline__ cplx<T> rot(cplx<T> a) {
  constexpr int k = ((K % M) * (16 / M)) & 15;
  if constexpr (k == 0) {
    return a;
  } else if constexpr (k == 8) {
    return {-a.x, -a.y};
  } else if constexpr ((k == 4 && DIR < 0) || (k == 12 && DIR > 0)) {
    return {a.y, -a.x};  // * (-i)
  } else if constexpr (k == 4 || k == 12) {
    return {-a.y, a.x};  // * (+i)
  } else {
    return ConstMul<T>::template mul<k, DIR, EXACT>(a);
  }
}

// Radix-2 decimation-in-frequency butterflies of one stage of length L at offset OFF.
template <int DIR, int L, int OFF, int I, bool EXACT, typename T>
struct DifStage {
  __device__ __forceinline__ static void run(cplx<T>* v) {
    if constexpr (I < L / 2) {
      cplx<T> a = v[OFF + I], b = v[OFF + I + L / 2];
      v[OFF + I] = cadd(a, b);
      v[OFF + I + L / 2] = rot<DIR, I, L, EXACT>(csub(a, b));
      DifStage<DIR, L, OFF, I + 1, EXACT, T>::run(v);
    }
  }
};
template <int DIR, int L, int OFF, bool EXACT, typename T>
struct Dif {
  __device__ __forceinline__ static void run(cplx<T>* v) {
    if constexpr (L > 1) {
      DifStage<DIR, L, OFF, 0, EXACT, T>::run(v);
      Dif<DIR, L / 2, OFF, EXACT, T>::run(v);
      Dif<DIR, L / 2, OFF + L / 2, EXACT, T>::run(v);
    }
  }
};

// In-register r-point DFT:  y_q = sum_j x_j exp(DIR*2*pi*i*j*q/r), r | 16.
template <int DIR, int r, bool EXACT, typename T>
__device__ __forceinline__ void dft(cplx<T>* x) {
  Dif<DIR, r, 0, EXACT, T>::run(x);
  cplx<T> y[r];
#pragma unroll
  for (int q = 0; q < r; ++q) y[q] = x[bitrev(q, ilog2(r))];
#pragma unroll
  for (int q = 0; q < r; ++q) x[q] = y[q];
}

// LDS index with one pad slot every PR entries (PR = the team's radix): spreads
// the radix-strided writes of a pass over the banks.
template <int PR>
__device__ __forceinline__ int padr(int i) { return i + i / PR; }
template <int N, int PR>
struct Padded {
  static constexpr int size = N + N / PR + 1;
};

// Padding of a column's LDS array of N + N/R entries where C columns are transposed between the load
// layout (C columns x consecutive rows in a wave) and wave teams: the C columns of a row then start
// 256 / C bytes apart in the 64 banks (with one entry, four columns met in the same banks: a third of
// the LDS cycles of a 512^2 sweep).
template <typename E, int C>
constexpr int col_pad() {
  constexpr int p = 256 / int(sizeof(cplx<E>)) / C;
  return p > 1 ? p : 1;
}

// LDS views of one team's working array.  ptr(pb) is the address of padded
// index pb; S is the element stride between consecutive padded indices.  The element
// type E may be narrower than the arithmetic type: exchanged values are then rounded
// to E (complex64 exchanges of an FP64 transform halve the LDS bytes).
template <typename E>
struct LdsRow {  // contiguous: a[i] at base[padr(i)]
  using elem = E;
  static constexpr int S = 1;
  cplx<E>* base;
  __device__ __forceinline__ cplx<E>* ptr(int pb) const { return base + pb; }
};
template <typename E, int LS>
struct LdsStrided {  // interleaved columns: a[i] at base[padr(i) * LS]
  using elem = E;
  static constexpr int S = LS;
  cplx<E>* base;
  __device__ __forceinline__ cplx<E>* ptr(int pb) const { return base + pb * LS; }
};

// complex conversion between arithmetic and LDS element types (identity when equal)
template <typename D, typename T>
__device__ __forceinline__ cplx<D> ccvt(cplx<T> v) {
  if constexpr (std::is_same_v<D, T>) {
    return v;
  } else {
    return {D(v.x), D(v.y)};
  }
}

// Hides the value of an expression from the optimiser, so that per-lane
// addresses and indices of one transform are not merged with (and kept live
// until) those of the next transform in the same kernel.
template <typename P>
__device__ __forceinline__ P opaque_s(P p) {
  asm volatile("" : "+s"(p));
  return p;
}
__device__ __forceinline__ int opaque_v(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Twiddle tables: FP64 hi only; FP32 hi and lo (the rounding error of hi).
template <typename T>
struct Twiddles {
  const cplx<T>* hi;
  const cplx<T>* lo;
};

// x * w (DIR < 0) or x * conj(w) (DIR > 0); FP32 adds the product with the low part l.
template <int DIR>
__device__ __forceinline__ cplx<double> tw_apply(cplx<double> x, cplx<double> w) {
  if (DIR > 0) w.y = -w.y;
  return cmul(x, w);
}
template <int DIR>
__device__ __forceinline__ cplx<float> tw_apply(cplx<float> x, cplx<float> w, cplx<float> l) {
  if (DIR > 0) {
    w.y = -w.y;
    l.y = -l.y;
  }
  const float rx = fmaf(x.x, w.x, -x.y * w.y), ry = fmaf(x.x, w.y, x.y * w.x);
  return {rx + fmaf(x.x, l.x, -x.y * l.y), ry + fmaf(x.x, l.y, x.y * l.x)};
}

template <int DIR>
__device__ __forceinline__ cplx<double> tw_mul(cplx<double> x, const Twiddles<double>& tw, int idx) {
  return tw_apply<DIR>(x, gload(gmem(tw.hi) + idx));
}
template <int DIR>
__device__ __forceinline__ cplx<float> tw_mul(cplx<float> x, const Twiddles<float>& tw, int idx) {
  return tw_apply<DIR>(x, gload(gmem(tw.hi) + idx), gload(gmem(tw.lo) + idx));
}

// Twiddles of every pass of one lane, held in registers for the whole kernel (a lane's
// twiddles depend only on its team index t, so all transforms of a sweep share them and
// the inverse uses their conjugates).  Only butterfly mm = 0 of a pass is stored: the
// passes before the last have one butterfly per lane (r = R), and in the last pass
// (span Ns = N / r, twiddle w^(j b), b = t + mm TT) butterfly mm differs from mm = 0 by
// the exact constant w^(j mm TT) = exp(-2 pi i j mm / R).  Slot of (pass P, input j >= 1):
// off(P) + j - 1.
template <int N, int R>
struct TwSlots {
  static constexpr int NP = num_passes(N, R);
  static constexpr int off(int P) {
    int o = 0;
    for (int q = 1; q < P; ++q) o += pass_radix(N, R, q) - 1;
    return o;
  }
  static constexpr int count = off(NP) > 0 ? off(NP) : 1;
};

// EXACT: transforms with them take the low part of sqrt(1/2) (ConstMul).
template <typename T, int N, int R, bool EXACT = false>
struct TwRegs;
template <int N, int R, bool EXACT>
struct TwRegs<double, N, R, EXACT> {
  static constexpr bool kExact = EXACT;
  cplx<double> hi[TwSlots<N, R>::count];
  template <int DIR>
  __device__ __forceinline__ cplx<double> mul(cplx<double> x, int slot, int) const {
    return tw_apply<DIR>(x, hi[slot]);
  }
  __device__ __forceinline__ void set(int slot, const Twiddles<double>& tw, int idx) { hi[slot] = gload(gmem(tw.hi) + idx); }
};
template <int N, int R, bool EXACT>
struct TwRegs<float, N, R, EXACT> {
  static constexpr bool kExact = EXACT;
  cplx<float> hi[TwSlots<N, R>::count], lo[TwSlots<N, R>::count];
  template <int DIR>
  __device__ __forceinline__ cplx<float> mul(cplx<float> x, int slot, int) const {
    return tw_apply<DIR>(x, hi[slot], lo[slot]);
  }
  __device__ __forceinline__ void set(int slot, const Twiddles<float>& tw, int idx) {
    hi[slot] = gload(gmem(tw.hi) + idx);
    lo[slot] = gload(gmem(tw.lo) + idx);
  }
};

// Table-backed source with the same interface (twiddle index idx, slot unused).
template <typename T, bool EXACT = false>
struct TwMem {
  static constexpr bool kExact = EXACT;
  Twiddles<T> tw;
  template <int DIR>
  __device__ __forceinline__ cplx<T> mul(cplx<T> x, int, int idx) const {
    return tw_mul<DIR>(x, tw, idx);
  }
};

// Fills the registers of team index t from the table.
template <typename T, int N, int R, int P = 1, bool EXACT = false>
__device__ __forceinline__ void load_twiddles(TwRegs<T, N, R, EXACT>& w, int t, const Twiddles<T>& tw) {
  if constexpr (P < num_passes(N, R)) {
    constexpr int r = pass_radix(N, R, P), Ns = ipow(R, P);
    const int tstep = (t % Ns) * (N / (Ns * r));
#pragma unroll
    for (int j = 1; j < r; ++j) w.set(TwSlots<N, R>::off(P) + j - 1, tw, (j * tstep) & (N - 1));
    load_twiddles<T, N, R, P + 1>(w, t, tw);
  }
}

// Calls f(std::integral_constant<int, i>) for i = B .. E-1.
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// Ordering of a pass's LDS write and read.  BlockSync: the team spans several waves.
// WaveSync: every lane of the team is in one wave, whose LDS operations execute in
// program order, so only the compiler has to keep the order (no s_barrier); the
// fences name the LDS address space only, so global loads (tables, twiddles) may
// still be scheduled across an exchange.
struct BlockSync {
  __device__ __forceinline__ static void sync() { __syncthreads(); }
};
struct WaveSync {
  __device__ __forceinline__ static void sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  }
};

// One Stockham pass P >= 1 (LDS-sourced) through the team's LDS view.
//
// Every LDS address is a per-lane base plus a compile-time offset: spans after
// the first pass are multiples of R, so padr(i + R m) = padr(i) + (R+1) m, and
// the first pass (radix R, span 1) writes the R consecutive indices of one
// aligned group of R, so padr(R b + q) = padr(R b) + q.
template <int BIT, typename T>
__device__ __forceinline__ void lane_swap(cplx<T>& a, cplx<T>& b);
template <typename T, int N, int R, int P>
struct PassIO {
  static constexpr int NP = num_passes(N, R);
  static constexpr int TT = N / R;
  // write the outputs of pass P-1 (team index t, strided register layout of that pass)
  template <class Lds>
  __device__ __forceinline__ static void write(const cplx<T> (&v)[R], int tl, Lds lds) {
    constexpr int rp = pass_radix(N, R, P - 1);  // radix of the previous pass
    constexpr int Nsp = ipow(R, P - 1);          // span before the previous pass
    constexpr int nbp = R / rp;
    constexpr int S = Lds::S;
    using E = typename Lds::elem;
    static_assert(Nsp % R == 0 || (Nsp == 1 && rp == R), "separable LDS offsets");
#pragma unroll
    for (int mm = 0; mm < nbp; ++mm) {
      const int b = tl + mm * TT;
      const int k = b % Nsp;
      cplx<E>* p = lds.ptr(padr<R>((b - k) * rp + k));
#pragma unroll
      for (int q = 0; q < rp; ++q) {
        constexpr int unit = Nsp == 1 ? 1 : Nsp / R * (R + 1);
        p[S * q * unit] = ccvt<E>(v[mm * rp + q]);
      }
    }
  }
  // read the inputs of pass P, twiddle, r-point DFTs; outputs in v
  template <int DIR, class Lds, class Tw>
  __device__ __forceinline__ static void read(cplx<T> (&v)[R], int tl, Lds lds, const Tw& tw) {
    constexpr int r = pass_radix(N, R, P);
    constexpr int Ns = ipow(R, P);
    constexpr int nb = R / r;
    constexpr int S = Lds::S;
    static_assert((N / r) % R == 0, "separable LDS offsets");
    static_assert(nb == 1 || P == NP - 1, "several butterflies per lane only in the last pass");
    static_assert(nb == 1 || Ns == N / r, "the last pass spans N / r");
    cplx<T> o[R];
    // twiddle of input j: w^(j k s), k = b mod Ns, s = N / (Ns r); for mm > 0 (last pass,
    // k = t + mm TT, s = 1) it is w^(j t) * exp(DIR 2 pi i j mm / R)
    const int tstep = (tl % Ns) * (N / (Ns * r));
    static_for<0, nb>([&](auto MM) {
      constexpr int mm = decltype(MM)::value;
      const auto* p = lds.ptr(padr<R>(tl + mm * TT));
      cplx<T> x[r];
#pragma unroll
      for (int j = 0; j < r; ++j) x[j] = ccvt<T>(p[S * j * ((N / r) / R * (R + 1))]);
      static_for<1, r>([&](auto J) {
        constexpr int j = decltype(J)::value;
        x[j] = tw.template mul<DIR>(x[j], TwSlots<N, R>::off(P) + j - 1, (j * tstep) & (N - 1));
        x[j] = rot<DIR, (j * mm) % R, R, Tw::kExact>(x[j]);
      });
      dft<DIR, r, Tw::kExact>(x);
      if constexpr (P == NP - 1) {
        // last pass: outputs land on t + TT*(mm + q*nb) -> strided register layout
#pragma unroll
        for (int q = 0; q < r; ++q) o[mm + q * nb] = x[q];
      } else {
#pragma unroll
        for (int q = 0; q < r; ++q) o[mm * r + q] = x[q];
      }
    });
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = o[j];
  }
  // the last pass with its inputs exchanged between lanes instead of through LDS (swaps_lanes):
  // register q = r mm + j then holds input j of butterfly t + mm TT
  template <int DIR, class Tw>
  __device__ __forceinline__ static void swap(cplx<T> (&v)[R], int tl, const Tw& tw) {
    constexpr int r = pass_radix(N, R, P), nb = R / r;
    constexpr int top = ilog2(TT) - 1;  // lane bit of the highest bit of j
    static_for<0, ilog2(r)>([&](auto B) {
      constexpr int bit = decltype(B)::value;  // bit of j
      static_for<0, R>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        if constexpr (!((q >> bit) & 1)) lane_swap<top - (ilog2(r) - 1 - bit)>(v[q], v[q | (1 << bit)]);
      });
    });
    cplx<T> o[R];
    static_for<0, nb>([&](auto MM) {
      constexpr int mm = decltype(MM)::value;
      cplx<T> x[r];
#pragma unroll
      for (int j = 0; j < r; ++j) x[j] = v[mm * r + j];
      static_for<1, r>([&](auto J) {
        constexpr int j = decltype(J)::value;
        x[j] = tw.template mul<DIR>(x[j], TwSlots<N, R>::off(P) + j - 1, (j * tl) & (N - 1));
        x[j] = rot<DIR, (j * mm) % R, R, Tw::kExact>(x[j]);
      });
      dft<DIR, r, Tw::kExact>(x);
#pragma unroll
      for (int q = 0; q < r; ++q) o[mm + q * nb] = x[q];
    });
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = o[j];
  }
};

// Exchange of a lane-index bit with a register-index bit: lane halves (BIT 5) or odd and even
// rows of 16 lanes (BIT 4) of the registers a (bit clear) and b (bit set).  Afterwards a holds
// what was in the lanes with the bit clear (of a, then of b), b what was in the others.
template <int BIT>
__device__ __forceinline__ void lane_swap(unsigned& a, unsigned& b) {
  static_assert(BIT == 4 || BIT == 5, "v_permlane16_swap_b32, v_permlane32_swap_b32");
  if constexpr (BIT == 5) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  }
}
template <int BIT, typename T>
__device__ __forceinline__ void lane_swap(cplx<T>& a, cplx<T>& b) {
  constexpr int W = sizeof(cplx<T>) / 4;
  struct Words {
    unsigned w[W];
  };
  Words x = __builtin_bit_cast(Words, a), y = __builtin_bit_cast(Words, b);
#pragma unroll
  for (int i = 0; i < W; ++i) lane_swap<BIT>(x.w[i], y.w[i]);
  a = __builtin_bit_cast(cplx<T>, x);
  b = __builtin_bit_cast(cplx<T>, y);
}

// The exchange before the last pass can stay in registers: lane t of a team holds the outputs q
// of butterfly t, whose top log2(r) index bits are the inputs j of the last pass, and the last
// pass needs lane bits and the low bits of q exchanged -- one swap instruction per register pair
// and bit where those are lane bits 4 and 5 (r = 4 on 64 lanes, r = 2 on 64 or 32 lanes).
// The LDS pipe of a CU serves its four SIMDs: an exchange of four radix-16 FP64 teams at N = 1024
// keeps it for about 1000 cycles while the FP64 units wait; the 64 swaps of a lane run on each
// SIMD by itself.  Measured (1024^2): damped FP64 step 52.7 -> 51.0 us, 32 FP64 grids 586 -> 565 us
// per step, 64 uneven complex64-state grids 275 -> 267 us.  Other lane bits have no swap
// instruction (moves through DPP need two to four per pair): those passes stay in LDS.
template <int N, int R, int P, class Sync>
constexpr bool swaps_lanes() {
  constexpr int r = pass_radix(N, R, P), TT = N / R;
  return std::is_same_v<Sync, WaveSync> && P == num_passes(N, R) - 1 && P >= 2 && r <= R && TT / r >= 16 &&
         (TT == 64 || TT == 32);
}

template <typename T, int N, int R, int DIR, int P, class Sync, class Lds, class Tw>
struct TeamPass {
  __device__ __forceinline__ static void run(cplx<T> (&v)[R], int t, Lds lds, const Tw& tw) {
    if constexpr (P < num_passes(N, R) && swaps_lanes<N, R, P, Sync>()) {
      PassIO<T, N, R, P>::template swap<DIR>(v, opaque_v(t), tw);
    } else if constexpr (P < num_passes(N, R)) {
      const int tl = opaque_v(t);
      Sync::sync();  // every lane has read the previous pass's inputs
      PassIO<T, N, R, P>::write(v, tl, lds);
      Sync::sync();
      PassIO<T, N, R, P>::template read<DIR>(v, tl, lds, tw);
      TeamPass<T, N, R, DIR, P + 1, Sync, Lds, Tw>::run(v, t, lds, tw);
    }
  }
};

// Full length-N transform by a team.  In/out: v[j] = a[t + j*TT] (natural order).
// lds: view of the team's private LDS array (Padded<N,R>::size entries).
// BlockSync contains __syncthreads(): every lane of the block must call it.
template <typename T, int N, int R, int DIR, class Lds, class Sync = BlockSync, class Tw = TwMem<T>>
__device__ __forceinline__ void team_fft(cplx<T> (&v)[R], int t, Lds lds, const Tw& tw) {
  static_assert(N % R == 0 && R <= 16 && (R & (R - 1)) == 0 && N >= R, "radix");
  dft<DIR, R, Tw::kExact>(v);  // pass 0: butterfly b = t reads v[j] = a[t + j*TT], no twiddle
  TeamPass<T, N, R, DIR, 1, Sync, Lds, Tw>::run(v, t, lds, tw);
}
template <typename T, int N, int R, int DIR, class Lds>
__device__ __forceinline__ void team_fft(cplx<T> (&v)[R], int t, Lds lds, Twiddles<T> tw) {
  team_fft<T, N, R, DIR, Lds, BlockSync, TwMem<T>>(v, t, lds, TwMem<T>{tw});
}

// Transform whose lanes change teams at the first exchange: the input is held in a
// load layout (team index tw_, LDS view lw of its team), the output in a compute layout
// (team index tc, view lc) whose teams each sit in one wave.  The first exchange is
// block-wide, every later one wave-local.  Every lane of the block must call it.
template <typename T, int N, int R, int DIR, class Lds, class Tw>
__device__ __forceinline__ void team_fft_remap(cplx<T> (&v)[R], int tl, Lds lw, int tc, Lds lc, const Tw& tw) {
  static_assert(num_passes(N, R) >= 2, "the remap happens at the first exchange");
  dft<DIR, R, Tw::kExact>(v);
  PassIO<T, N, R, 1>::write(v, opaque_v(tl), lw);
  __syncthreads();
  const int t = opaque_v(tc);
  PassIO<T, N, R, 1>::template read<DIR>(v, t, lc, tw);
  TeamPass<T, N, R, DIR, 2, WaveSync, Lds, Tw>::run(v, tc, lc, tw);
}

}  // namespace wh
