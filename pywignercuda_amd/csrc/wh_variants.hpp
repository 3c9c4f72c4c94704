// Launch variants of the fused sweeps: (radix R, lanes per block).  The tuner
// (pywignercuda_amd/tune.py) times the valid variants per grid size on the GPU
// and stores its choice; the host falls back to the first valid entry.
#pragma once

namespace wh {

// tp: throughput form for batches of grids: twiddles read from the table instead of
// held in registers and the exchanges between transform passes held in the state's
// storage precision (complex64 for the complex64-state FP64-arithmetic form), so that
// three waves fit per SIMD (<= 168 VGPRs, ~36-41 KiB of LDS per block)
struct SweepVariant {
  int R, block, tp;
};

// index 0 is the default.  The entries behind the first kNumX, kNumP, kNumPCL are narrow forms: a plan
// takes one in place of the 256-lane form of its radix where its cells give that fewer blocks than
// the chip has CUs (kCUs).  A block's exchanges share its CU's LDS pipe, so that a few wide blocks
// wait for the LDS while other CUs are idle: the damped 128^2 step, 8 blocks of 256 lanes, takes 18.1
// us, 32 blocks of 64 take 15.4; 256^2 18.9 and 15.7; 512 x 256 21.0 and 18.1.  Where 256-lane blocks
// fill the CUs they are faster (whole 64-byte rows: 1024 x 512 31.6, with 128 lanes 33.9), and of the
// narrow forms the widest that fills them (512^2: 23.6 with 256 lanes, 21.7 with 128, 22.8 with 64).
constexpr SweepVariant kXVariants[] = {{16, 256, 0}, {8, 256, 0}, {8, 512, 0}, {4, 256, 0}, {16, 256, 1}, {8, 64, 0}, {4, 64, 0}};
constexpr SweepVariant kPVariants[] = {{16, 256, 0}, {8, 512, 0}, {8, 256, 0}, {16, 256, 1}, {8, 128, 0}, {8, 64, 0}};
constexpr SweepVariant kPCLVariants[] = {{16, 256, 0}, {8, 256, 0}, {16, 256, 1}, {8, 128, 0}, {8, 64, 0}};
constexpr int kAllX = sizeof(kXVariants) / sizeof(kXVariants[0]), kNumX = kAllX - 2;
constexpr int kAllP = sizeof(kPVariants) / sizeof(kPVariants[0]), kNumP = kAllP - 2;
constexpr int kAllPCL = sizeof(kPCLVariants) / sizeof(kPCLVariants[0]), kNumPCL = kAllPCL - 2;
constexpr int kCUs = 256;

// The Gross-Pitaevskii shift: rows of G in teams of one wave at most (radix 8, sides up to 512) where
// kGpWide's blocks would be fewer than the CUs.
constexpr SweepVariant kGpWide{16, 256, 0}, kGpNarrow{8, 64, 0};

// largest grid side of the plain (x and p) throughput forms
constexpr int kTpMaxN = 1024;

// same rule as size_ok<N, R, BLOCK>() in wh_sweeps.hpp (and the throughput forms' size bound,
// which the Caldeira-Leggett one does not have; cl: a Caldeira-Leggett p variant)
constexpr bool variant_fits(int N, SweepVariant v, bool cl = false) {
  return N >= v.R * 4 && N / v.R <= v.block && v.block / (N / v.R) <= 64 && (!v.tp || cl || N <= kTpMaxN);
}
// rows per x-sweep tile / columns per p-sweep tile
constexpr int tile_lines(int N, SweepVariant v) { return v.block / (N / v.R); }

// the x variants of a Gross-Pitaevskii plan: the default (index 0) has at least as many rows per tile as
// the two others it may be created with, at every side (its partial density sums fit their buffer)
constexpr bool default_fits_partials() {
  for (int N = 128; N <= 2048; N *= 2)
    for (int v : {1, 3})
      if (!variant_fits(N, kXVariants[0]) || tile_lines(N, kXVariants[0]) < tile_lines(N, kXVariants[v])) return false;
  return true;
}
static_assert(default_fits_partials(), "partial density sums");

}  // namespace wh
