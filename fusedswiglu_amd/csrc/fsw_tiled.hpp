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
  double us;                    // the estimate
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
  Plan best{8, 1, steps, 0, 0, 1, steps, 1e30};
  auto consider = [&](Plan p, double us) {
    p.us = us;
    if (us < best.us) best = p;
  };
  for (int mb = 8; mb >= 4; mb--) {
    const long long tile_m = C::kTileM * mb / 8, tiles_m = (M + tile_m - 1) / tile_m, tiles = tiles_m * tiles_n;
    consider(Plan{mb, 1, steps, 0, 0, 1, steps, 0}, std::max(rounds_us(tiles, steps, mb, tiles_m), bytes / 5.5e6));
    if (C::kForward) continue;
    // splits that leave the chip a third, half or two thirds full (fewer partial tiles) or fill it once, twice or three
    // times; at least 8 steps per workgroup
    for (long long sixths : {2, 3, 4, 6, 12, 18}) {
      const long long s = std::min({sixths * kCus / 6 / tiles, (long long)steps / 8, 64LL});
      if (s < 2) continue;
      const SplitPlan sp = split_steps(steps, (int)s);
      if (sp.splits < 2 || (double)sp.splits * elems * 4 > (double)ws_bytes) continue;
      consider(Plan{mb, sp.splits, sp.steps_per_split, 0, 0, 1, steps, 0},
               std::max(rounds_us(tiles * sp.splits, sp.steps_per_split, mb, tiles_m), bytes / 5.5e6) + 5.8 + sp.splits * elems * 8 / 6.9e6);
    }
    const TailPlan t = plan_tail(tiles, steps);
    if (mb == 8 && t.count > 0 && tail_bytes(t) <= ws_bytes)
      consider(Plan{mb, 1, steps, t.first, t.count, t.parts, t.steps, 0},
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
  return Plan{8, sp.splits, sp.steps_per_split, 0, 0, 1, steps, 0};
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

// Whether the four-wave form can address the operands: it walks an m/n-contiguous one through 32-bit offsets from its first
// k-row.  Larger ones take the eight-wave form (256-row tiles).
template <int MODE>
bool fits_four_waves(const GemmParams& g) {
  using C = Cfg<MODE>;
  return (C::kAKc || (long long)g.K * g.lda * 2 < (1LL << 31)) && (C::kBKc || (long long)g.K * g.ldb * 2 < (1LL << 31));
}
template <int MODE>
Lines lines_of(const GemmParams& g) { return Lines{whole_lines(g.lda), whole_lines(g.ldb)}; }

// Returns the workgroups of the launch.
template <int MODE>
long long set_plan(GemmParams& g, const Plan& p, void* ws) {
  using C = Cfg<MODE>;
  const int tile_m = C::kTileM * p.mb / 8;
  g.tiles_m = (g.M + tile_m - 1) / tile_m;
  g.tiles_n = (g.N + C::kTileN - 1) / C::kTileN;
  // Height of the bands of tile-rows an XCD walks (band_tile).  The A panels of the 8 bands in
  // flight (8 XCDs x group_m panels of 256 rows x K) should stay in the 256 MB memory-side cache while
  // the B panels stream past: 8 tile-rows up to K = 4096, 4 beyond (measured at K = 8192: 4 % faster).
  g.group_m = g.K > 4096 ? 4 : 8;
  g.ws = (float*)ws; g.splits = p.splits; g.steps_per_split = p.steps_per_split;
  g.tail_first = p.tail_first; g.tail_count = p.tail_count; g.tail_parts = p.tail_parts; g.tail_steps = p.tail_steps;
  const long long tiles = (long long)g.tiles_m * g.tiles_n;
  g.split_per_xcd = split_per_xcd(tiles * p.splits, p.steps_per_split);
  return p.tail_count > 0 ? p.tail_first + (long long)p.tail_count * p.tail_parts : tiles * p.splits;
}

template <typename E, int MODE>
hipError_t launch_typed(GemmParams g, hipStream_t s, void* ws, long long ws_bytes) {
  using C = Cfg<MODE>;
  const bool fits = fits_four_waves<MODE>(g);
  const Plan p = fits ? plan<MODE>(g.M, g.N, g.K, ws ? ws_bytes : 0, lines_of<MODE>(g)) : plan_eight_waves<MODE>(g.M, g.N, g.K, ws ? ws_bytes : 0);
  const long long grid = set_plan<MODE>(g, p, ws);
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

// ---- both gradients in one launch -----------------------------------------------------------------------------------
// The weight and the input gradient wait for the same gating gradients, and on problems of a few rounds each alone leaves much
// of its last round empty: at 8192 x 256 x 768 156 and 64 workgroups on 256 CUs, one after the other.  In one launch the second
// GEMM's workgroups start on the CUs that the first leaves, higher tiles (which cost less per row) fill the chip together, and
// start, end and the sum of partial planes are paid once.  The whole backward behind a forward, gating gradient included, two
// launches -> one: 8192 x 256 x 768 54.3 -> 43.9 us, 2048 x 512 x 1536 50.8 -> 37.5, 2048 x 1024 x 2736 80.5 -> 65.1, 8192 x 1024 x
// 3072 223 -> 204; 120 random steps of 256 to 32768 tokens, d_model 256 to 8192: 0.89 of the time on average, 0.59 the best.
// Large problems, whose last round is a small part of the launch, stay at two launches (plan_pair's margin).  The two gradients
// of the down projection wait for the same operand as well.
// The operands of a gradient GEMM from a Problem; mode kDw / kDwT and kDx / kDxT by the layout of the weights.
inline GemmParams weight_grad_params(const Problem& p) {
  GemmParams g{};
  if (p.w_out_in) {  // dWg [I,D] = dG^T x: the two results share the B tile (x)
    g.a0 = p.dG; g.a1 = p.dU; g.b0 = p.x; g.c0 = p.dWg; g.c1 = p.dWu;
    g.M = (int)p.I; g.N = (int)result_cols(p.D); g.n_rows_b = (int)p.D; g.K = (int)p.T;
    g.lda = (int)p.ldo; g.ldb = (int)p.ldx; g.ldc = (int)p.lddw;
    return g;
  }
  g.a0 = p.x; g.b0 = p.dG; g.b1 = p.dU; g.c0 = p.dWg; g.c1 = p.dWu;
  g.M = (int)p.D; g.N = (int)result_cols(p.I); g.n_rows_b = (int)p.I; g.K = (int)p.T;
  g.lda = (int)p.ldx; g.ldb = (int)p.ldo; g.ldc = (int)p.lddw;
  return g;
}
inline GemmParams input_grad_params(const Problem& p) {
  GemmParams g{};
  g.a0 = p.dG; g.a1 = p.dU; g.b0 = p.wg; g.b1 = p.wu; g.c0 = p.dx;
  g.M = (int)p.T; g.N = (int)result_cols(p.D); g.n_rows_b = (int)p.D; g.K = (int)p.I;
  g.lda = (int)p.ldo; g.ldb = (int)p.ldw; g.ldc = (int)p.lddx;
  return g;
}

inline GemmParams gemm_params(const GemmProblem& p) {
  GemmParams g{};
  g.a0 = p.a; g.b0 = p.b; g.c0 = p.c;
  g.M = (int)p.M; g.N = (int)result_cols(p.N); g.n_rows_b = (int)p.N; g.K = (int)p.K;
  g.lda = (int)p.lda; g.ldb = (int)p.ldb; g.ldc = (int)p.ldc;
  return g;
}

struct PairPlan {
  Plan w, x;      // w.mb == 0: two launches are better
  bool x_first;   // the longer workgroups first
  double us;
};
// Tile heights (16-row blocks per wave of w, of x) that the pair kernel is built for: of all 25 combinations these give up 1 %
// of the backward's time on average, four of them 2 % more.
constexpr int kPairHeights[][2] = {{8, 8}, {8, 4}, {4, 8}, {4, 4}, {5, 5}, {7, 8}, {8, 7}};

// Microseconds of na workgroups of ta each and, behind them, nb of tb each, tb <= ta, on all CUs: a workgroup starts on the
// first CU that is free.
inline double two_jobs_us(long long na, double ta, long long nb, double tb) {
  const long long late = na % kCus, early = kCus - late;  // CUs that are free after `full` rounds of a, and one round later
  const double t_early = na / kCus * ta, t_late = t_early + ta;
  if (nb == 0) return late ? t_late : t_early;
  // each early CU takes e workgroups of b and each late one l: the smallest end that has room for nb
  long long e = std::max(0LL, nb / kCus - 1);
  for (;; e++) {
    const double end = t_early + e * tb;
    const long long l = end > t_late ? (long long)((end - t_late) / tb) : 0;
    if (e * early + l * late >= nb) return std::max(end, late ? t_late : 0.0);
    const double end_late = t_late + (l + 1) * tb;  // before the early CUs end another one
    if (late && end_late < end + tb && e * early + (l + 1) * late >= nb) return std::max(end_late, t_late);
  }
}

// Bytes of a plan's fp32 partial planes.
template <int MODE>
double plane_bytes(const Plan& p, const GemmParams& g) {
  return p.splits > 1 ? 4.0 * p.splits * Cfg<MODE>::kResults * g.M * g.N : 0.0;
}

// What a GEMM by itself would be offered of scratch that is there for two: workspace_of, which asks for the plan of dense rows.
// Where rows are not whole lines apart, plan() would take more parts than it asked for if it had the scratch.
template <int MODE>
long long scratch_for_one(const GemmParams& g, long long ws_bytes) {
  const Lines here = lines_of<MODE>(g), dense = dense_lines<MODE>(g.M, g.N, g.K);
  if (here.a == dense.a && here.b == dense.b) return ws_bytes;
  return std::min(ws_bytes, workspace_of<MODE>(g.M, g.N, g.K));
}

template <int MODE_W, int MODE_X>
PairPlan plan_pair(const GemmParams& w, const GemmParams& x, long long ws_bytes) {
  PairPlan none{}, best{};
  const Lines lw = lines_of<MODE_W>(w), lx = lines_of<MODE_X>(x);
  // The splits are those of two launches, so that a sum is made of the same parts in either case.
  const Plan pw = plan<MODE_W>(w.M, w.N, w.K, scratch_for_one<MODE_W>(w, ws_bytes), lw);
  const Plan px = plan<MODE_X>(x.M, x.N, x.K, scratch_for_one<MODE_X>(x, ws_bytes), lx);
  if (pw.tail_count > 0 || px.tail_count > 0) return none;
  const double planes = plane_bytes<MODE_W>(pw, w) + plane_bytes<MODE_X>(px, x);
  if (planes > (double)ws_bytes) return none;
  best.us = 0.97 * (pw.us + px.us + 1.0);  // (a predicted gain below that came out between -3 and +1 %)
  const double reduce = planes > 0 ? 5.8 + planes * 2 / 6.9e6 : 0.0;
  for (const auto& mb : kPairHeights) {
    const long long rows_w = Cfg<MODE_W>::kTileM * mb[0] / 8, rows_x = Cfg<MODE_X>::kTileM * mb[1] / 8;
    const long long tm_w = (w.M + rows_w - 1) / rows_w, tm_x = (x.M + rows_x - 1) / rows_x;
    const long long nw = tm_w * ((w.N + Cfg<MODE_W>::kTileN - 1) / Cfg<MODE_W>::kTileN) * pw.splits;
    const long long nx = tm_x * ((x.N + Cfg<MODE_X>::kTileN - 1) / Cfg<MODE_X>::kTileN) * px.splits;
    const double tw = pw.steps_per_split * step_us<MODE_W>(mb[0], 1.0, tm_w, lw) + 1.3 + 0.68 * mb[0];
    const double tx = px.steps_per_split * step_us<MODE_X>(mb[1], 1.0, tm_x, lx) + 1.3 + 0.68 * mb[1];
    const double work = (nw * tw + nx * tx) / kCus;
    if (work + reduce >= best.us || nw + nx > (1LL << 30)) continue;
    const double end = tx > tw ? two_jobs_us(nx, tx, nw, tw) : two_jobs_us(nw, tw, nx, tx);
    const double us = end * (0.7 + 0.3 * work / end) + reduce;
    if (us < best.us) {
      best = PairPlan{pw, px, tx > tw, us};
      best.w.mb = mb[0];
      best.x.mb = mb[1];
    }
  }
  return best;
}

// Scratch for the partial planes of both in one launch, 0 if they would not share one.
template <int MODE_W, int MODE_X>
long long pair_workspace(const GemmParams& w, const GemmParams& x) {
  if (!fits_four_waves<MODE_W>(w) || !fits_four_waves<MODE_X>(x)) return 0;
  const PairPlan pl = plan_pair<MODE_W, MODE_X>(w, x, 1LL << 62);
  return pl.w.mb == 0 ? 0 : (long long)(plane_bytes<MODE_W>(pl.w, w) + plane_bytes<MODE_X>(pl.x, x));
}

template <typename E, int MODE_W, int MODE_X, int I = 0>
void launch_pair_kernel(const PairParams& p, int mb_w, int mb_x, unsigned grid, hipStream_t s) {
  if constexpr (I < (int)(sizeof(kPairHeights) / sizeof(kPairHeights[0]))) {
    constexpr int W = kPairHeights[I][0], X = kPairHeights[I][1];
    if (mb_w == W && mb_x == X) fsw_gemm4_pair_kernel<E, MODE_W, W, MODE_X, X><<<grid, kThreads4, 0, s>>>(p);
    else launch_pair_kernel<E, MODE_W, MODE_X, I + 1>(p, mb_w, mb_x, grid, s);
  }
}

// *done: whether the pair took the launch; if not, nothing has been enqueued.
template <typename E, int MODE_W, int MODE_X>
hipError_t launch_pair(GemmParams w, GemmParams x, hipStream_t s, void* ws, long long ws_bytes, bool* done) {
  *done = false;
  if (!fits_four_waves<MODE_W>(w) || !fits_four_waves<MODE_X>(x)) return hipSuccess;
  const PairPlan pl = plan_pair<MODE_W, MODE_X>(w, x, ws ? ws_bytes : 0);
  if (pl.w.mb == 0) return hipSuccess;
  PairParams p{};
  const size_t floats_w = (size_t)plane_bytes<MODE_W>(pl.w, w) / 4;
  p.w_count = (int)set_plan<MODE_W>(w, pl.w, ws);
  p.x_count = (int)set_plan<MODE_X>(x, pl.x, (float*)ws + floats_w);
  p.w = w;
  p.x = x;
  p.w_first = pl.x_first ? (p.x_count + 7) & ~7 : 0;
  p.x_first = pl.x_first ? 0 : (p.w_count + 7) & ~7;
  const unsigned grid = (unsigned)std::max(p.w_first + p.w_count, p.x_first + p.x_count);
  *done = true;
  launch_pair_kernel<E, MODE_W, MODE_X>(p, pl.w.mb, pl.x.mb, grid, s);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || (w.splits == 1 && x.splits == 1)) return e;
  auto blocks = [](const GemmParams& g) { return g.splits > 1 ? (unsigned)(((size_t)g.M * g.N / 4 + 255) / 256) : 0u; };
  fsw_pair_reduce_kernel<E, Cfg<MODE_W>::kResults><<<Cfg<MODE_W>::kResults * blocks(w) + blocks(x), 256, 0, s>>>(p, (int)blocks(w));
  return hipGetLastError();
}

// The pairs in float16: each is instantiated in another file than the same pair in bfloat16, so that no file takes all of the
// compiler's time.
hipError_t launch_grads_pair_fp16(const Problem& p, hipStream_t s, void* ws, long long ws_bytes, bool* done);
hipError_t launch_gemm_pair_fp16(const GemmParams& w, const GemmParams& x, int layout, hipStream_t s, void* ws, long long ws_bytes, bool* done);

}  // namespace fsw
