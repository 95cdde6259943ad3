// How the weight-streaming kernels (at most 128 rows) cut a problem into workgroups: host arithmetic only.
#pragma once
#include <algorithm>

namespace fsw {

// Width of a workgroup's column block.  128 columns fill the LDS slot, but a launch is one workgroup per block
// and every block takes the same time, so what counts is rounds x width: the width that covers N with the
// fewest rounds of `cus` workgroups wins (I = 28672 on 256 CUs: 256 blocks of 112 instead of 224 of 128;
// I = 12288 and 16 rows: 256 blocks of 48 instead of 96 of 128).  Two limits, both measured:
//  * weights stored [D, I] are read in row segments that must start on 128-byte lines (partial lines are
//    fetched whole, by two workgroups): widths of 64 and 128 only; rows of [I, D] weights are lines of
//    their own: any multiple of 8;
//  * a narrower block leaves part of every 32 KiB weight slot empty while the x rows stay, so the useful
//    bytes in flight per CU shrink: not below 48 / 64 / 96 columns for up to 32 / 64 / 128 rows.
inline int block_width(int N, int cus, bool w_kc, int bm) {
  const int step = w_kc ? 8 : 64;
  const int narrowest = w_kc ? (bm <= 32 ? 48 : (bm <= 64 ? 64 : 96)) : 64;
  int best = 128;
  long long best_cost = (long long)(((N + 127) / 128 + cus - 1) / cus) * 128;
  for (int bn = 128 - step; bn >= narrowest; bn -= step) {
    const long long cost = (long long)(((N + bn - 1) / bn + cus - 1) / cus) * bn;
    if (cost < best_cost) { best = bn; best_cost = cost; }
  }
  return best;
}

// A launch: column blocks of `slot` = 128 (fsw_skinny_forward_kernel) or 16, 32, 64 columns (fsw_narrow_kernel; mq
// 16-row blocks of x), of which bn are used, times k-splits.  paired: 8 columns whose gate and up rows share a slot of 16.
struct SkPlan { int slot, mq, bn, splits, stages_per_split; bool paired; };
// k-elements of a stage of the narrow kernel (NarrowCfg)
inline int narrow_stage(int slot, int mq, bool paired, long long M) { return paired ? (M <= 8 ? 256 : 128) : slot == 16 || (slot == 32 && mq == 1) ? 128 : 64; }

// Blocks of 128 columns for the down projection: full blocks and as many k-splits as fit into one round of workgroups
// (measured at N = 8192, K = 28672: 32 blocks x 8 splits beat every narrower block with fewer splits in this kernel,
// although the partial planes then cost 2 x 8 x M x N x 4 bytes of traffic: narrow blocks leave the 32 KiB weight slots
// half empty).  Enough column blocks for a round on their own, or the forward: no split, and the width rule above.
inline SkPlan plan_wide(long long M, long long Nh, long long K, int cus, bool w_kc, long long max_splits) {
  const int stages = (int)((K + 63) / 64);
  const long long tiles = (Nh + 127) / 128;
  // a split shorter than 8 stages does not fill the ring
  const long long splits = std::min({cus / tiles, max_splits, (long long)stages / 8});
  if (max_splits < 1 || splits <= 1) return SkPlan{128, 0, block_width((int)Nh, cus, w_kc, (int)M), 1, stages, false};
  const int sps = (int)((stages + splits - 1) / splits);
  return SkPlan{128, 0, 128, (stages + sps - 1) / sps, sps, false};
}

// Microseconds of a launch by what it moves, fitted to 9700 measured launches with weights that are not in the caches (1 to
// 128 rows, d_model 1024 .. 8192, d_intermediate 2 .. 4 times that, both layouts, forward and down projection; rms error
// 10 %): all weights once at 6 TB/s; per CU its weights at 49 (128-column blocks: 26) bytes/ns and its LDS fill, x
// included, at 50 (62) bytes/ns; start and end of a launch and of every further round of workgroups; the second launch of a
// split and its fp32 partials.  Rows of [D, I] weights shorter than a 128-byte line are fetched as whole lines by every
// block.  128-column blocks in parts, up to 16 rows, [I, D], cost more than that fit knows: 0.2 us for the start of each part, and
// where rows of the weights start between lines 10 % more for the weights, whose row segments then share lines.  With both, and
// with `rows` of choose_within for every narrow block of such a product, 3 x 382 down projections of 1 to 16 rows, 1024 to 9400
// columns and reductions of 1024 to 28672 take 1.010 of what the best of the forms takes, 1.039 before: 1 x 8704 -> 3568 16.0 -> 12.6
// us, 10 x 8584 -> 8048 41.2 -> 29.9, 6 x 4088 -> 7984 22.3 -> 15.5; 8 of them take 1.03 to 1.10 of their time before, all of 16 rows
// or below 11 us (16 x 14336 -> 3456 22.3 -> 24.1).
inline double estimate_us(const SkPlan& p, long long M, long long Nh, long long K, int cus, bool w_kc) {
  const bool wide = p.slot == 128;
  const long long wgs = (Nh + p.bn - 1) / p.bn * p.splits, rounds = (wgs + cus - 1) / cus;
  const int x_rows = p.paired && M <= 8 ? 8 : !wide ? 16 * p.mq : (M <= 32 ? 32 : (M <= 64 ? 64 : 128));
  const double stage = wide ? 64 : narrow_stage(p.slot, p.mq, p.paired, M);
  const double k64 = (double)rounds * p.stages_per_split * stage / 64;  // 64-element blocks a CU goes through
  const double lines = w_kc || p.slot >= 64 ? 1 : 64 / p.slot;
  const double useful = k64 * p.bn * 256 * lines, fill = k64 * (256 * (p.paired ? p.bn : p.slot) * lines + 128 * x_rows);
  const double cu_rate = w_kc ? (wide ? 26e3 : 49e3) : (wide ? 30e3 : 36e3), fill_rate = w_kc ? (wide ? 62e3 : 50e3) : (wide ? 55e3 : 47e3);
  const double start = w_kc ? (wide ? 0.6 : 4.2) : (wide ? 1.2 : 4.3), round = wide ? 2.0 : (w_kc ? 1.3 : 0.0);
  double us = std::max({4.0 * K * Nh / 6.0e6, useful / cu_rate, fill / fill_rate}) + start + round * (rounds - 1);
  if (p.splits > 1) us += (w_kc ? 1.7 : 2.3) + p.splits * M * Nh * 8.0 / 1.3e6;
  if (wide && p.splits > 1 && w_kc && M <= 16) us += 0.2 * p.splits + (K % 64 ? 0.1 * 4.0 * K * Nh / 6.0e6 : 0.0);
  return us;
}

// Nh: columns of each half.  Narrow blocks are taken where the estimate sees them ahead by more than it errs among the
// launches above, whose times they then beat on average by 31 / 23 / 28 / 21 % (forward, [I, D], up to 16 / 32 / 64 / 128
// rows), 15 / 16 / 19 / 15 % (down projection, nn.Linear's layout), 5 / 2 / 4 / 12 % and 10 / 9 / 2 / 0 % (the other
// layout): 1 x 1024 x 3072 [I, D] 10.5 -> 5.6 us, 16 x 2048 x 4096 17.6 -> 9.1, 1 x 4096 x 11008
// 36.9 -> 33.2, the down projection of 64 x 2048 x 4096 15.4 -> 10.9.  [D, I] weights of more than 150 MB stay on blocks of 128: their rows, one
// segment per k and block, are then read 15 to 20 % slower in shorter segments.
// Outside those launches: whole_lines says that the rows of the weights are a multiple of 128 bytes apart (only the
// forward's plan asks).  Where the rows of [I, D] weights start between lines, a forward of up to 32 rows stays on blocks of 128 once
// 32-column blocks need a second round: 64-column blocks then read 4.2 TB/s and the 48 of 128 up to 5 (60 launches of 1 to 32
// rows, 8200 to 11808 columns: narrow blocks took 1.10 to 1.21 of the time in all but one, 0.99 in that; 1 x 5448 x 11704
// 60.7 -> 51.3 us).  More rows, one round of 32-column blocks, or the down projections: narrow blocks win there between lines
// as well.  What is left: a down projection of more than 64 rows with more than 40 MB of weights, reduction contiguous.  The
// estimate errs both ways there, narrow blocks took 0.84 to 1.24 of the time (geometric mean 1.0), and no simple rule parts them.
// 8-column blocks whose gate and up rows share the 16 rows of an MFMA operand ([I, D], up to 16 rows; NarrowCfg): twice the
// workgroups of 16-column blocks and no half-empty slots, and a result of up to 4096 columns needs neither parts nor the launch
// that adds them: 1 / 8 / 16 x 11008 -> 4096 21.1 / 21.5 / 22.3 us in 16 parts of 128 columns, 18.9 / 19.7 / 21.6 so; 1 x 8704 -> 4096
// 17.4 and 13.9.  A second round of them is longer than wider blocks (1 x 8704 -> 4112 20.8 us, 32 columns in parts 17.0).
// A forward takes them where a width that fills its rounds comes to 8 columns (1032 to 2048 columns; to 4400 in two rounds): 0.76 of the
// time of the narrow form without them in 105 random ones, worst 0.92 (1 x 1240 x 1792 6.9 -> 5.2 us, 16 x 8536 x 1064 27.5 -> 18.8).
inline SkPlan choose_within(long long M, long long Nh, long long K, int cus, bool w_kc, bool whole_lines, bool plain,
                            long long max_splits) {
  SkPlan best = plan_wide(M, Nh, K, cus, w_kc, plain ? max_splits : 0);
  if (!w_kc && 4.0 * K * Nh > 150e6) return best;
  if (w_kc && !plain && !whole_lines && M <= 32 && Nh > 32LL * cus) return best;
  double best_us = estimate_us(best, M, Nh, K, cus, w_kc);
  best_us /= plain ? (M <= 16 ? 1.05 : 1.15) : (w_kc ? 1.10 : 1.0);
  // x rows that are there cost more than those that zero-fill (12 x 5440 -> 1984 10.3 us, paired 10.9; 6 x 9472 -> 2560 13.8 and 14.6)
  const bool few = w_kc && plain && M <= 16;
  const double rows = M <= 4 ? 1.0 : M <= 8 ? 1.04 : 1.08;
  for (int slot = 16; slot <= (w_kc ? 64 : 32); slot *= 2) {
    int mq = slot == 64 ? 2 : 1;
    while (16 * mq < M) mq *= 2;
    // a third round of 16-column blocks: 1 to 29 % longer than blocks of 64 or 128 in 11 of 12 down projections of up to 16 rows
    // (16 x 7232 -> 17536 56.3 -> 43.6 us; 6 x 7760 -> 17520 67.0 -> 69.7)
    if (slot == 16 && (mq > 4 || (w_kc && Nh > 32LL * cus))) continue;
    // widths: the whole slot; rows of [I, D] weights are lines of their own, so also what fills 1 .. 5 rounds, and 8
    // columns for short results
    for (int i = 0; i <= (w_kc ? 6 : 0); i++) {
      const int bn = i == 0 ? slot : (i == 6 ? 8 : (int)(((Nh + cus * i - 1) / (cus * i) + 3) & ~3LL));
      const bool paired = w_kc && bn == 8 && mq == 1;
      if (bn > slot || bn < slot / 2 || (i == 6 && !plain)) continue;
      const int stage = narrow_stage(slot, mq, paired, M), stages = (int)((K + stage - 1) / stage);
      const long long blocks = (Nh + bn - 1) / bn;
      for (int splits : {1, 2, 3, 4, 6, 8}) {
        // (8-column blocks in parts: no faster than whole in 40 of 42 launches, for all their scratch and the second launch)
        if (splits > 1 && (!plain || paired || splits > max_splits || blocks * splits > 560 || K < 128 * splits)) break;
        if (blocks * splits < (splits > 1 ? 48 : 40)) continue;
        const int sps = (stages + splits - 1) / splits;
        const SkPlan pl{slot, mq, bn, (stages + sps - 1) / sps, sps, paired};
        const double us = estimate_us(pl, M, Nh, K, cus, w_kc) * (paired || few ? rows : 1.0);
        if (us < best_us) { best_us = us; best = pl; }
      }
    }
  }
  return best;
}

// Splits of a reduction that scratch for any number of planes may have.
constexpr long long kSkMaxSplits = 16;

// The launch for scratch of max_splits fp32 planes.  What the workspace query asks for, the plan under no limit, is taken
// whenever its planes fit.  A search under a limit only finds it by chance: 8 parts of 18 stages are 6 parts of 3, but 6 as a
// limit rules out 8, and an unsplit plan has won against a split one of 128-column blocks that a call without scratch does
// not weigh.  One shape in 14 took another plan than the one its scratch was sized for, and 10 % more time on average
// (50 such shapes): the down projection of 119 x 1280 -> 448 19.3 instead of 9.5 us, of 26 x 1280 -> 256 12.1 instead of 7.8.
inline SkPlan choose(long long M, long long Nh, long long K, int cus, bool w_kc, bool whole_lines, bool plain,
                     long long max_splits) {
  const SkPlan p = choose_within(M, Nh, K, cus, w_kc, whole_lines, plain, kSkMaxSplits);
  return !plain || p.splits <= max_splits ? p : choose_within(M, Nh, K, cus, w_kc, whole_lines, plain, max_splits);
}

}  // namespace fsw
