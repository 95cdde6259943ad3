// Host side of the tiled MFMA kernels: the plan of a launch and the launch itself.
#pragma once
#include "fsw_gemm.hpp"
#include "fsw_gemm4.hpp"
#include "fsw_internal.hpp"
#include <algorithm>

namespace fsw {

// ---- how a problem is cut into workgroups ---------------------------------------------------------------------
// A launch is rounds of 256 workgroups (one per CU), and every workgroup of a round takes the same time.  Three things
// can be chosen so that the rounds are full and short: how many rows a tile has (32 mb, mb = 4 .. 8 blocks of 16 per
// wave: 128 .. 256 rows; kDwT half of that per result), over how many workgroups the reduction of a tile is split
// (gradients and plain GEMMs: fp32 partial tiles in the caller's scratch, added up by a second kernel in a fixed order),
// and whether only the tiles of a short last round are split.  plan() takes the cheapest by an estimate of the time:
//   round     steps * step_us[mb] + 1.3 + 0.68 mb us (pipeline fill, epilogue);
//             a last round of r workgroups: its steps at 0.7 + 0.3 r/256 of that (the chip is power limited)
//   split     5.8 us (second launch, its latency) + 8 bytes per partial element at 6.9 TB/s
//   floor     operands and results once at 5.5 TB/s
// step_us and what lengthens it are given below.
// The constants are fitted to 6086 measured launches on operands that are not in the caches (six modes, 46 shapes of 129 ..
// 16384 tokens, d_model 256 .. 8192, every mb and up to 24 splits; fit within 8 %): the plan found is on average 1 %
// behind the best of those measured.  Against whole tiles of 256 rows only (same shapes, operands cached): forward 20 %,
// dx 18 %, dW 15 % faster on average; 777 x 4096 x 11008 forward 160 -> 123 us (160-row tiles), 2048 x 2048 x 5632
// forward 97 -> 80 and dW 95 -> 83 us (192 rows), 200 x 4096 x 11008 forward 72 -> 52 us (128 rows).
struct Plan {
  int mb;                       // 16-row blocks per wave
  int splits, steps_per_split;  // splits == 1: whole reduction
  int tail_first, tail_count, tail_parts, tail_steps;  // tail split (GemmParams); tail_count == 0: off
};

constexpr long long kCus = 256;

struct SplitPlan { int splits, steps_per_split; };
inline SplitPlan split_steps(int steps, int splits) {
  int sps = (steps + splits - 1) / splits;
  sps = (sps + 1) & ~1;  // pairs of steps stay together
  const int n = (steps + sps - 1) / sps;
  return n > 1 ? SplitPlan{n, sps} : SplitPlan{1, steps};
}

// Tail split: when the tiles do not fill the last round of 256 workgroups, each tile of that round goes to
// `parts` workgroups that reduce a slice each (fsw_gemm.hpp, GemmParams).  Only for long reductions and at
// least one full round before; the partial tiles take count * parts * 256 KiB of scratch.
struct TailPlan { int first, count, parts, steps; };
inline TailPlan plan_tail(long long tiles, int steps) {
  TailPlan t{0, 0, 1, steps};
  const int count = (int)(tiles % kCus);
  if (tiles < kCus || count == 0 || count > 128 || steps < 128) return t;
  int parts = 256 / count;
  if (parts > 8) parts = 8;
  if (parts > steps / 32) parts = steps / 32;
  if (parts < 2) return t;
  const SplitPlan sp = split_steps(steps, parts);
  t.first = (int)(tiles - count);
  t.count = count;
  t.steps = sp.steps_per_split;
  t.parts = sp.splits;
  return t;
}
inline long long tail_bytes(const TailPlan& t) { return (long long)t.count * t.parts * kTileFloats * 4; }

// Scratch a caller is asked for: enough to split the reduction until whole tiles fill the chip (as far as that pays at
// 1 us per step and 4 TB/s for the partial tiles), or to split the tail.  Plans take what is offered, up to this or to
// what plan() wants on top.
inline SplitPlan scratch_splits(long long tiles, int steps, double result_elems) {
  if (tiles >= 1024 || steps < 32) return SplitPlan{1, steps};
  auto cost = [&](int s) {
    const double rounds = (double)((tiles * s + kCus - 1) / kCus);
    return rounds * ((double)steps / s + 6.0) * 0.96 + (s > 1 ? 2.0 * s * result_elems * 4.0 / 4.0e6 : 0.0);
  };
  int best = 1;
  double best_cost = cost(1);
  const int max_s = steps / 16 < 64 ? steps / 16 : 64;
  for (int s = 2; s <= max_s; s++) {
    const double c = cost(s);
    if (c < best_cost * 0.95) { best_cost = c; best = s; }
  }
  return split_steps(steps, best);
}

inline int steps_of(int mode, long long K) {
  int steps = (int)((K + kBK - 1) / kBK);
  return (mode == kDx || mode == kDxT) ? 2 * ((steps + 1) & ~1) : steps;
}

// Whether the rows of A and B are a whole number of 128-byte lines apart.  (Of their pitch alone: where a tensor starts does not
// change the order of a sum.)
struct Lines { bool a, b; };
inline bool whole_lines(long long ld) { return (ld & 63) == 0; }
// Dense operands: the pitch of each is its contiguous dimension.
template <int MODE>
Lines dense_lines(long long M, long long N, long long K) {
  return Lines{whole_lines(result_cols(Cfg<MODE>::kAKc ? K : M)), whole_lines(result_cols(Cfg<MODE>::kBKc ? K : N))};
}

// Microseconds of one 32-element step with 16 mb rows per wave, `fill` of the CUs at work (1: all of them, power limited).
// The loads of a step take longer, and low tiles, which have the most of them per row, lose what they gain,
//  * where the rows of an operand are not whole lines: the 128-byte (KC) or 256-byte (MC) piece of a row touches one more;
//  * with a single row of tiles: no other workgroup reads the same piece of B, all of it comes from HBM.
// Without these two the plan was more than 10 % behind the best of all heights and splits at 5.1 % of 6180 problems of up to
// 160 rows and at 3.2 % of 16144 larger ones whose rows are not whole lines; with them at 2.4 and 1.6 % (whole lines, 48136
// problems: 0.8 % either way).  Input gradients of 90 x 8184 x 26856 314 -> 202 us, 122 x 8064 x 19776 184 -> 145, 4182 x 1608 x
// 3288 120 -> 101.  (A table of its own for kDwT at mb = 4, whose rings are shorter, helps operands that are not cached and
// costs a training step, where they are, 2 to 3 %.)
template <int MODE>
inline double step_us(int mb, double fill, long long tiles_m, Lines lines) {
  using C = Cfg<MODE>;
  constexpr double forward[5] = {0.435, 0.500, 0.588, 0.650, 0.720};
  constexpr double kc_a[5] = {0.431, 0.483, 0.564, 0.618, 0.673};   // kDx*, kNN, kNT
  constexpr double mc_a[5] = {0.428, 0.508, 0.562, 0.638, 0.692};   // kDw*, kTN
  double us = (C::kForward ? forward : C::kAKc ? kc_a : mc_a)[mb - 4] * (0.7 + 0.3 * fill);
  if (tiles_m == 1) us = std::max(us, mb <= 5 ? 0.34 + 0.30 * fill : 0.45 + 0.26 * fill);
  if (C::kAKc && !lines.a) us += 0.0125 * mb;
  if (!lines.b) us += C::kBKc ? 0.1 : 0.045;
  return us;
}

template <int MODE>
Plan plan(long long M, long long N, long long K, long long ws_bytes, Lines lines) {
  using C = Cfg<MODE>;
  const int steps = steps_of(MODE, K);
  const long long tiles_n = (N + C::kTileN - 1) / C::kTileN;
  const double elems = (double)M * N * C::kResults;
  const double bytes = 2.0 * ((double)M * K * (C::kPasses * (C::kDualM ? 2 : 1)) + (double)N * K * (C::kPasses * (C::kDualN ? 2 : 1)) +
                              elems * (C::kForward ? 3 : 1));
  auto rounds_us = [&](long long wgs, int s, int mb, long long tiles_m) {
    const double edge = 1.3 + 0.68 * mb;
    const long long full = wgs / kCus, rest = wgs % kCus;
    return (full ? full * (s * step_us<MODE>(mb, 1.0, tiles_m, lines) + edge) : 0.0) +
           (rest ? s * step_us<MODE>(mb, (double)rest / kCus, tiles_m, lines) + edge : 0.0);
  };
  Plan best{8, 1, steps, 0, 0, 1, steps};
  double best_us = 1e30;
  auto consider = [&](const Plan& p, double us) {
    if (us < best_us) { best_us = us; best = p; }
  };
  for (int mb = 8; mb >= 4; mb--) {
    const long long tile_m = C::kTileM * mb / 8, tiles_m = (M + tile_m - 1) / tile_m, tiles = tiles_m * tiles_n;
    consider(Plan{mb, 1, steps, 0, 0, 1, steps}, std::max(rounds_us(tiles, steps, mb, tiles_m), bytes / 5.5e6));
    if (C::kForward) continue;
    // splits that leave the chip a third, half or two thirds full (fewer partial tiles) or fill it once, twice or three
    // times; at least 8 steps per workgroup
    for (long long sixths : {2, 3, 4, 6, 12, 18}) {
      const long long s = std::min({sixths * kCus / 6 / tiles, (long long)steps / 8, 64LL});
      if (s < 2) continue;
      const SplitPlan sp = split_steps(steps, (int)s);
      if (sp.splits < 2 || (double)sp.splits * elems * 4 > (double)ws_bytes) continue;
      consider(Plan{mb, sp.splits, sp.steps_per_split, 0, 0, 1, steps},
               std::max(rounds_us(tiles * sp.splits, sp.steps_per_split, mb, tiles_m), bytes / 5.5e6) + 5.8 + sp.splits * elems * 8 / 6.9e6);
    }
    const TailPlan t = plan_tail(tiles, steps);
    if (mb == 8 && t.count > 0 && tail_bytes(t) <= ws_bytes)
      consider(Plan{mb, 1, steps, t.first, t.count, t.parts, t.steps},
               rounds_us(t.first, steps, mb, tiles_m) + rounds_us((long long)t.count * t.parts, t.steps, mb, tiles_m) + 5.8 + tail_bytes(t) * 2 / 6.9e6);
  }
  return best;
}

// The eight-wave form has tiles of 256 rows (kDwT 128) only and takes the split that scratch was asked for, or none: its
// operands span 2^31 bytes along the reduction, so few tiles mean a reduction of thousands of steps for each.  Weight
// gradients of 131072 x 256 x 8192, 524288 x 1024 x 2048 and 2097152 x 256 x 768: 1.1, 3.5 and 1.9 ms split, 2.5, 9.6 and
// 38 ms on whole tiles.
template <int MODE>
Plan plan_eight_waves(long long M, long long N, long long K, long long ws_bytes) {
  using C = Cfg<MODE>;
  const int steps = steps_of(MODE, K);
  const long long tiles = ((M + C::kTileM - 1) / C::kTileM) * ((N + C::kTileN - 1) / C::kTileN);
  SplitPlan sp{1, steps};
  if (!C::kForward) sp = scratch_splits(tiles, steps, (double)M * N * C::kResults);
  if (sp.splits > 1 && (double)sp.splits * M * N * 4 * C::kResults > (double)ws_bytes) sp = SplitPlan{1, steps};
  return Plan{8, sp.splits, sp.steps_per_split, 0, 0, 1, steps};
}

// Scratch for a GEMM of the given mode with results `results` x [M, N] and a reduction of K per pass.  with_tail: as a
// caller is told, enough for whatever plan() may choose and for padded rows; without, the split reduction alone.
template <int MODE>
long long workspace_of(long long M, long long N, long long K, bool with_tail = true) {
  using C = Cfg<MODE>;
  if (with_tail) N = result_cols(N);
  const long long tiles = ((M + C::kTileM - 1) / C::kTileM) * ((N + C::kTileN - 1) / C::kTileN);
  const int steps = steps_of(MODE, K);
  const long long plane = M * N * 4 * C::kResults;
  const int asked = scratch_splits(tiles, steps, (double)M * N * C::kResults).splits;
  if (!with_tail) return asked > 1 ? asked * plane : 0;
  const Plan p = plan<MODE>(M, N, K, 1LL << 62, dense_lines<MODE>(M, N, K));
  return std::max({asked > 1 ? asked * plane : 0LL, p.splits > 1 ? p.splits * plane : 0LL, asked > 1 ? 0LL : tail_bytes(plan_tail(tiles, steps))});
}

// Which slices of a split reduction an XCD works on.  All tiles of a slice read the same k-elements, so an XCD that has few
// slices and many of their tiles fetches far less into its L2 than one that has a few tiles of every slice: 16384 x 256 x 768
// weight gradient (12 tiles x 20 slices) with its reduce 34.0 -> 27.3 us, 1024 x 1024 x 4096 input gradient 31.0 -> 28.2, the
// down projection of 777 x 11008 -> 4096 83.1 -> 79.5.  Short slices that leave a fifth of the CUs or more without work are
// the exception: they are over before any rate counts, and tiles that all wait for the same lines at once take longer to
// start (120 random problems of 130 to 16384 tokens: 1 to 16 % longer in 26 of the 43 such, 1.03 on average; the other 77
// take 0.962, the worst of them 1.025).
inline bool split_per_xcd(long long workgroups, int steps) { return steps >= 24 || workgroups > 204; }

template <typename E, int MODE, bool STREAM>
void launch4(const GemmParams& g, int mb, unsigned grid, hipStream_t s) {
  switch (mb) {
    case 4: fsw_gemm4_kernel<E, MODE, 4, STREAM><<<grid, kThreads4, 0, s>>>(g); break;
    case 5: fsw_gemm4_kernel<E, MODE, 5, STREAM><<<grid, kThreads4, 0, s>>>(g); break;
    case 6: fsw_gemm4_kernel<E, MODE, 6, STREAM><<<grid, kThreads4, 0, s>>>(g); break;
    case 7: fsw_gemm4_kernel<E, MODE, 7, STREAM><<<grid, kThreads4, 0, s>>>(g); break;
    default: fsw_gemm4_kernel<E, MODE, 8, STREAM><<<grid, kThreads4, 0, s>>>(g); break;
  }
}

template <typename E, int MODE>
hipError_t launch_typed(GemmParams g, hipStream_t s, void* ws, long long ws_bytes) {
  using C = Cfg<MODE>;
  // The four-wave form walks an m/n-contiguous operand through 32-bit offsets from its first k-row; larger operands
  // take the eight-wave form (256-row tiles).
  const bool fits = (C::kAKc || (long long)g.K * g.lda * 2 < (1LL << 31)) && (C::kBKc || (long long)g.K * g.ldb * 2 < (1LL << 31));
  const Lines lines{whole_lines(g.lda), whole_lines(g.ldb)};
  const Plan p = fits ? plan<MODE>(g.M, g.N, g.K, ws ? ws_bytes : 0, lines) : plan_eight_waves<MODE>(g.M, g.N, g.K, ws ? ws_bytes : 0);
  const int tile_m = C::kTileM * p.mb / 8;
  g.tiles_m = (g.M + tile_m - 1) / tile_m;
  g.tiles_n = (g.N + C::kTileN - 1) / C::kTileN;
  // Height of the bands of tile-rows an XCD walks (xcd_tile_order).  The A panels of the 8 bands in
  // flight (8 XCDs x group_m panels of 256 rows x K) should stay in the 256 MB memory-side cache while
  // the B panels stream past: 8 tile-rows up to K = 4096, 4 beyond (measured at K = 8192: 4 % faster).
  g.group_m = g.K > 4096 ? 4 : 8;
  g.ws = (float*)ws; g.splits = p.splits; g.steps_per_split = p.steps_per_split;
  g.split_per_xcd = split_per_xcd((long long)g.tiles_m * g.tiles_n * p.splits, p.steps_per_split);
  g.tail_first = p.tail_first; g.tail_count = p.tail_count; g.tail_parts = p.tail_parts; g.tail_steps = p.tail_steps;
  const long long tiles = (long long)g.tiles_m * g.tiles_n;
  const long long grid = p.tail_count > 0 ? p.tail_first + (long long)p.tail_count * p.tail_parts : tiles * p.splits;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  // a forward with a single row of tiles reads every weight byte exactly once: stream them past the caches
  const bool stream = C::kForward && g.tiles_m == 1;
  if (fits) {
    if constexpr (C::kForward) {
      if (stream) launch4<E, MODE, true>(g, p.mb, (unsigned)grid, s);
    }
    if (!stream) launch4<E, MODE, false>(g, p.mb, (unsigned)grid, s);
  } else if constexpr (!(C::kAKc && C::kBKc)) {
    if constexpr (C::kForward) {
      if (stream) fsw_gemm_kernel<E, MODE, true><<<(unsigned)grid, kThreads, 0, s>>>(g);
    }
    if (!stream) fsw_gemm_kernel<E, MODE><<<(unsigned)grid, kThreads, 0, s>>>(g);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if constexpr (!C::kForward) {
    if (g.tail_count > 0) {
      fsw_tail_reduce_kernel<E, MODE><<<dim3((unsigned)(kTileFloats / 8192), (unsigned)g.tail_count), 256, 0, s>>>(g);
      return hipGetLastError();
    }
  }
  if (p.splits == 1) return e;
  const size_t n = (size_t)g.M * g.N;
  fsw_splitk_reduce_kernel<E><<<dim3((unsigned)((n / 4 + 255) / 256), (unsigned)C::kResults), 256, 0, s>>>(
      (const float*)ws, (unsigned short*)g.c0, (unsigned short*)g.c1, n, p.splits, g.N, g.ldc);
  return hipGetLastError();
}

template <int MODE>
hipError_t launch(int dtype, const GemmParams& g, hipStream_t s, void* ws = nullptr, long long ws_bytes = 0) {
  return dtype == kDtypeBF16 ? launch_typed<BF16, MODE>(g, s, ws, ws_bytes) : launch_typed<FP16, MODE>(g, s, ws, ws_bytes);
}

}  // namespace fsw
