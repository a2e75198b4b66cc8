// Mapping of work-group ids to (slice, block) for the attention kernels; plain
// C++ so that a host program can check it exhaustively.
#ifndef FMHA_BLOCK_MAP_H_
#define FMHA_BLOCK_MAP_H_

#if defined(__HIPCC__)
#define FMHA_HOST_DEVICE __host__ __device__ inline
#define FMHA_HOST __host__
#else
#define FMHA_HOST_DEVICE inline
#define FMHA_HOST
#endif

// A divisor that is the same for a whole launch.  A kernel divides by it with a multiplication, an addition and a shift; a
// division by an int is a chain of some 40 instructions, 250 cycles in which the work group has nothing else to do, and to
// find its block and its rows takes three to five of them.  Where a work group spends a few thousand cycles on its tiles that
// counts: figures at FmhaOrder.  Good for 0 <= n < 2^31: with mul = floor(2^32 (2^shift - d) / d) + 1, 2^32 + mul exceeds 2^(32 +
// shift) / d by at most 1, hence the quotient n (2^32 + mul) / 2^(32 + shift) exceeds n / d by less than 1 / d
// (Granlund and Montgomery, Division by Invariant Integers using Multiplication, 1994).
struct FmhaDivisor {
  int d;
  unsigned mul, shift;
  FmhaDivisor() = default;
  FMHA_HOST FmhaDivisor(int by) : d(by), shift(0) {
    while ((1ull << shift) < (unsigned long long)by) ++shift;
    mul = (unsigned)((((1ull << shift) - (unsigned long long)by) << 32) / (unsigned long long)by + 1);
  }
  FMHA_HOST_DEVICE operator int() const { return d; }
};
FMHA_HOST_DEVICE int operator/(int n, const FmhaDivisor& by) {
  const unsigned high = (unsigned)(((unsigned long long)(unsigned)n * by.mul) >> 32);
  return (int)((high + (unsigned)n) >> by.shift);
}

// Work-group id -> (batch*head slice, block inside the slice).  Consecutive
// work-group ids go round-robin over the 8 XCDs, each with a private L2; the
// remap hands every XCD whole (batch, head) slices, so the blocks that stream
// the same K/V (or Q/dO) rows share one L2.  An XCD takes its slices in groups
// of kSlicesInFlight: inside a group the blocks are ordered block-index major,
// and callers number blocks heaviest first, so under causal masking the heavy
// blocks of a group start before its light ones while the rows being streamed
// at any time (kSlicesInFlight slices) stay within the 4 MiB L2.
// When the slice count is no multiple of 8, the slices / 8 (rounded down)
// slices per XCD are handled as above by the first work-group ids; the blocks
// of the remaining slices % 8 slices follow in slice-major order, cut into 8
// contiguous runs, one per XCD, so that each of those slices is shared by as
// few XCDs as possible.
#ifndef FMHA_SLICES_IN_FLIGHT
#define FMHA_SLICES_IN_FLIGHT 2
#endif
constexpr int kSlicesInFlight = FMHA_SLICES_IN_FLIGHT;
template <typename Int>  // int or FmhaDivisor
FMHA_HOST_DEVICE void fmha_slice_and_block(int lin, int slices, const Int& blocks_per_slice, int& slice, int& blk) {
  const int q = slices >> 3, r = slices & 7;
  const int main_blocks = 8 * q * blocks_per_slice;
  if (lin < main_blocks) {
    const int xcd = lin & 7, slot = lin >> 3;  // slot: 0 .. q * blocks_per_slice - 1 inside the XCD
    const int group = slot / kSlicesInFlight / blocks_per_slice, within = slot - group * (kSlicesInFlight * blocks_per_slice);
    const int first = group * kSlicesInFlight;
    const int g = (q - first < kSlicesInFlight ? q - first : kSlicesInFlight);  // slices in this group
    blk = g == kSlicesInFlight ? within / kSlicesInFlight : kSlicesInFlight == 2 ? within : within / g;
    slice = xcd * q + first + (within - blk * g);
  } else {
    const int rem = lin - main_blocks, n_rem = r * blocks_per_slice;
    const int xcd = rem & 7, slot = rem >> 3;
    const int idx = xcd * (n_rem >> 3) + (xcd < (n_rem & 7) ? xcd : (n_rem & 7)) + slot;  // position in the slice-major list
    const int s = idx / blocks_per_slice;
    slice = 8 * q + s;
    blk = idx - s * blocks_per_slice;
  }
}

// Persistent launches: G work groups (one per CU) share the `total` blocks numbered as above.
// Work group w takes, in round r, block r * G + w for even r and r * G + (w mirrored inside its
// XCD, i.e. among the work groups congruent to w modulo 8) for odd r.  Both keep the block number
// congruent to w modulo 8, so the block stays on w's XCD, and the alternation pairs the heavy
// blocks of one round with the light blocks of the next (blocks are numbered heaviest first).
// G must be a multiple of 8 unless the launch has a single round (total <= G).
// fmha_persistent_block: the block of work group w in round r; >= total means none.
// fmha_persistent_next_round: the next round after r in which w has a block, or -1.
FMHA_HOST_DEVICE int fmha_persistent_block(int r, int w, int G) {
  const int p = (r & 1) ? (((G >> 3) - 1 - (w >> 3)) << 3) + (w & 7) : w;
  return r * G + p;
}
FMHA_HOST_DEVICE int fmha_persistent_next_round(int r, int w, int G, int total) {
  for (++r; (long)r * G < total; ++r)
    if (fmha_persistent_block(r, w, G) < total) return r;
  return -1;
}

// Whether the shares of G persistent work groups come out even.  Without a mask all blocks weigh the same: the last round
// has to be nearly full.  Under causal masking every work group has to get as many heavy blocks as light ones of the same
// slices, which takes whole pairs of rounds and whole slices for every XCD: the shares are then equal to the tile.  Pairs of
// rounds that are just nearly full are not enough: the largest share of 60 slices of 8 blocks (480 on 256 work groups) is
// 1.54 times the mean, of 42 slices of 12 blocks 1.8 times, of 120 slices of 8 blocks still 1.07 times.
FMHA_HOST_DEVICE bool fmha_even_shares(int slices, int blocks_per_slice, int G, bool causal) {
  const long total = (long)slices * blocks_per_slice;
  if (causal) return (slices & 7) == 0 && total % (2 * G) == 0;
  return total * 16 >= (total + G - 1) / G * G * 15;
}

// Whether the persistent 256-query forward takes a D = 128 problem.  It does up to 10 % more per second than the 128-query
// kernel where all CUs are busy, but a CU takes or leaves a whole block of 256.  Figures: us of the 128-query kernel, then of
// this one, at N x slices, over stretches of 0.15 s in turn.  The chip is at its power cap and what one kernel draws slows the
// others, so a call counts with what else runs: "+" with its backward behind.  Cards differ: A and B.
//   Under causal masking where its static shares come out even, whatever the number of rounds, from N = 4096 on, where a block
// has 32 tiles on average.  A: 4096 x 64 265, 261, + 1108, 1104; x 96 413, 399, + 1674, 1660; x 128 548, 541, + 2244, 2246; x
// 192 828, 806, + 3355, 3343; 6144 x 64 581, 565, + 2350, 2345; 8192 x 64 1012, 967, + 4081, 4032; x 96 1686, 1441, + 6458,
// 6207; x 128 2060, 1947, + 8249, 8178.  B: 4096 x 64 264, 247, + 1153, 1085; x 96 412, 384, + 1698, 1633; x 128 549, 514, +
// 2240, 2207; x 512 2164, 2063, + 8890, 8768; 8192 x 96 1641, 1397, + 6283, 5996; 8001 x 64 957, 923, + 3881, 3852; 16384 x
// 64 4104, 3518, + 15367, 14829.  In turns of 12 ms each has the clock that both together leave, which favours the one that
// draws more: 4096 x 96 397, 396; x 192 790, 809; 8192 x 128 1963, 1915.  Not at N = 2048, where card A shows nothing (x 64 76.2,
// 74.7, + 319, 323; x 128 148, 149, + 651, 653) though B does (x 128 147, 146, + 681, 646); nor with uneven shares: 4100 x
// 128 571, 669; 5120 x 64 415, 450; 7168 x 64 787, 890.
//   Without a mask, from N = 1152 on, where the last round of the 128-query kernel (two blocks to a CU, so that half a round
// costs it 0.6 of one) is more than half full and this one needs no more rounds.  A: 4096 x 16 126, 114, + 499, 488; x 64 485,
// 448, + 1974, 1945; x 25 (1.56 rounds) 220, 198, + 883, 888; x 42 (2.6) 343, 314, + 1356, 1346; 8192 x 13 434, 387, + 1722,
// 1700; 2048 x 30 (0.94) 64.3, 59.9, + 260, 258; 2048 x 64 129, 122, + 534, 530; 3000 x 20 90.1, 82.7, + 367, 365; 1500 x 42
// 51.9, 48.3, + 211, 210; 1500 x 69 (1.6) 89.7, 87.7, + 380, 386.  Not with half a round or less: the idle CUs leave the others
// a higher clock when nothing else runs, but not beside a backward that is at the cap.  4096 x 24 (1.5) 188, 197; x 56 (3.5)
// 428, 415, + 1736, 1748; x 68 (4.25) 530, 520, + 2173, 2187; x 100 (6.25) 779, 753, + 3191, 3192; 8192 x 28 (3.5) 842, 801,
// + 3337, 3369; x 42 (5.25) 1280, 1228, + 5118, 5166; 16384 x 17 (4.25) 2062, 1998, + 8134, 8289; 2048 x 168 (5.25) 361, 353,
// + 1440, 1451.  (B: 4096 x 56 + 1768, 1721; x 100 + 3165, 3148; 8192 x 42 + 4961, 4997.)  Nor where N is just past a multiple
// of 256: 1152 x 84 (1.5) 60.3, 71.3; 1031 x 120 (1.9; 2.3 of this kernel's) 82.8, 99.1.  Shorter sequences only where the last
// round is nearly full, as good alone, not with a backward: 1024 x 64 38.1, 36.2, + 154, 158; 512 x 128 24.1, 23.9, + 98, 103;
// 256 x 512 32.0, 30.8, + 139, 142; not 1024 x 224 (3.5) 121, 132.
constexpr int kPersistentForwardRows = 256;  // queries of a block
FMHA_HOST_DEVICE bool fmha_persistent_forward_pays(int slices, int n, int cus, bool causal) {
  const int blocks_per_slice = (n + kPersistentForwardRows - 1) / kPersistentForwardRows;
  if (causal) return n >= 4096 && fmha_even_shares(slices, blocks_per_slice, cus, true);
  if (n < 1152) return fmha_even_shares(slices, blocks_per_slice, cus, false);
  const long total = (long)slices * blocks_per_slice;
  const long rows = (long)slices * n, round = (long)cus * kPersistentForwardRows, left = rows % round;
  return (left == 0 || 2 * left > round) && (total + cus - 1) / cus <= (rows + round - 1) / round;
}

// Which MFMAs both passes of the D = 128 backward use, the same in both, since it decides the order of dS in the workspace: 16
// x 16 where the chip runs at its power cap, 32 x 32 where a good part of the CUs has nothing to do and a wave's own
// instructions are what takes the time.  fused_mha_backward has so few blocks only without a mask, from one for two CUs on:
// fewer, and all under causal masking, go in one launch, with 32 x 32 MFMAs (fmha_passes_at_once), unless the passes are
// called one by one.  us of the backward (statistics, both passes, dS stored) with 32 x 32 and with 16 x 16 MFMAs, N x slices
// (blocks per CU): without a mask 4096 x 2 (0.25) 125, 130; 1031 x 9 (0.32) 45.9, 46.7; 4096 x 4 (0.5) 132, 134; 1031 x 15
// (0.53) 47.1, 47.6; 1024 x 18 (0.56) 47.3, 46.8; 2048 x 9 76.6, 76.9; 1024 x 19 (0.59) 48.9, 47.9; 4096 x 5 (0.63) 145, 140;
// 2048 x 10 80.2, 78.3; 1031 x 20 (0.7) 52.9, 50.6; 512 x 64 (1) 43.8, 40.1; 1024 x 32 66.3, 59.7; 32 x 32 ahead by 0.7 % in
// the median of 11 more lengths between 0.5 and 0.63, by 0.4 % of 31 without room for dS (1439 x 13 75.2, 76.4).  Causal,
// where a block is half as much work: 8192 x 2 (0.5) 236, 246; 4096 x 6 (0.75) 134, 135; 2048 x 14 (0.88) 78.8, 79.5; 1031 x
// 28 (0.98) 52.5, 52.3; 2048 x 16 (1) 82.1, 82.2; 4096 x 8 147, 146; 2048 x 18 (1.13) 88.0, 86.3; 4096 x 10 (1.25) 163, 160;
// 4096 x 12 (1.5) 182, 176.
FMHA_HOST_DEVICE bool fmha_wide_mfmas(long key_blocks, int cus, bool causal) {  // blocks of 128 keys of a launch
  return causal ? key_blocks <= cus : 8 * key_blocks < 5L * cus;
}

// Launches of one block per work group that the hardware hands out as CUs become free, two or more to a CU.
// heavy_first (causal masking, blocks numbered heaviest first): the blocks of many slices are ordered block-index
// major, so that heavy blocks start first and the launch ends with light ones.  An XCD's slices are taken in groups of
// kScheduledSlices (the last group holds the rest too): groups of 8 instead of 2 took 3-19 % off the causal forward
// from N = 512 to 4096, 16 lost some of it again.  The rows that 8 slices stream fit the XCD's 4 MiB of L2 up to N =
// 1024 at D = 128; past that some are read again (dK/dV pass at B2 H32 N4096: 748 MB instead of 283 come from beyond
// the L2) for no time that could be measured: that pass is 1 % faster than with groups of 2, the dQ pass after it 2 %
// slower.  The slices % 8 that no XCD has for itself go one block per level to successive XCDs, in the last group.
// Otherwise (all blocks weigh the same) the order is fmha_slice_and_block's, except that with short_last the last block
// of every slice, which has fewer rows, comes at the end of the launch.
constexpr int kScheduledSlices = 8;
// `run`: the blocks of a slice that go in order (not its short last one); `last_level`: fmha_last_level.
template <typename Int>  // int or FmhaDivisor
FMHA_HOST_DEVICE void fmha_ordered_block(int lin, int slices, const Int& run, const Int& last_level, bool heavy_first,
                                         bool short_last, int& slice, int& blk) {
  if (!heavy_first) {
    if (!short_last || lin < slices * run) {
      fmha_slice_and_block(lin, slices, run, slice, blk);
    } else {
      slice = lin - slices * run;
      blk = run;
    }
    return;
  }
  const int q = slices >> 3;
  const int groups = q < kScheduledSlices ? 1 : q / kScheduledSlices;
  int group = lin / (8 * kScheduledSlices) / run;
  if (group > groups - 1) group = groups - 1;
  const int first = group * kScheduledSlices;
  const bool last = group == groups - 1;
  const int count = last ? q - first : kScheduledSlices;  // slices per XCD in this group
  const int level = last ? (int)last_level : 8 * kScheduledSlices;  // blocks of one index in this group
  const int idx = lin - 8 * first * run;
  blk = last ? idx / last_level : idx / (8 * kScheduledSlices);
  const int p = idx - blk * level;
  slice = (p >> 3) < count ? (lin & 7) * q + first + (p >> 3) : 8 * q + (p - 8 * count);
}
// Blocks of one index in the last group, which has the slices % 8 too.
FMHA_HOST_DEVICE int fmha_last_level(int slices) {
  const int q = slices >> 3, groups = q < kScheduledSlices ? 1 : q / kScheduledSlices;
  return slices - 8 * kScheduledSlices * (groups - 1);
}
FMHA_HOST_DEVICE int fmha_blocks_in_order(int blocks_per_slice, bool heavy_first, bool short_last) {
  return !heavy_first && short_last && blocks_per_slice > 1 ? blocks_per_slice - 1 : blocks_per_slice;
}
// This and the two like it below, fmha_two_pass_block and fmha_ds_launch_block, are for checks on the host: the same order from
// whole numbers, worked out anew for each block.  Kernels take an FmhaOrder.
FMHA_HOST_DEVICE void fmha_scheduled_block(int lin, int slices, int blocks_per_slice, bool heavy_first, bool short_last,
                                           int& slice, int& blk) {
  const int run = fmha_blocks_in_order(blocks_per_slice, heavy_first, short_last);
  fmha_ordered_block(lin, slices, run, fmha_last_level(slices), heavy_first, run < blocks_per_slice, slice, blk);
}

// The same launches, two blocks to a CU: work groups w and w + kCus start on the same CU, so with the second kCus taken in
// reverse (inside each XCD, which keeps a block on the XCD of its slice) a CU starts with one heavy and one light block
// instead of the k-th heaviest of either half.  Returns the position in the order above that work group `lin` takes.  us
// before and after, forward, then backward (D = 64, N x slices, blocks per CU): 512 x 128 (2) 14.2, 12.1; 38.3, 33.9.  1024 x
// 64 (2) 16.3, 15.5; 47.2, 45.6.  4096 x 16 (2) 48.6, 47.2; 154.8, 146.7.  1024 x 40 (1.25) 14.7, 14.5; 41.4, 41.0.  1024 x
// 66 17.8, 17.4; 50.1, 46.8.  1024 x 96 (3) 23.5, 23.1; 70.1, 66.4.  1024 x 128 (4) 30.5, 28.9; 87.1, 84.7.  8192 x 12 (3)
// 126, 124; 388, 382.  2048 x 64 (4) 45.4, 45.6; 141, 139.  Forward, D = 128: 1500 x 32 (1.5) 29.5, 27.9; 2048 x 80 (5) 95.6,
// 95.0.  Later blocks go where a place is free: the fourth kCus reversed as well loses (1024 x 128 29.6; 86.8).
constexpr int kCus = 256;  // of an MI355X; on any other number of CUs this is just another order
FMHA_HOST_DEVICE int fmha_paired_block(int lin, int total) {
  if (lin < kCus || lin >= 2 * kCus) return lin;
  const int xcd = lin & 7, end = total < 2 * kCus ? total : 2 * kCus;
  const int slots = (end - xcd + 7) >> 3;  // work groups below `end` on this XCD
  return ((kCus / 8 + slots - 1 - (lin >> 3)) << 3) + xcd;
}

// The 128-query forward where the last block of every slice has up to 32 queries: those of `per` (2 or 4) slices can go to one
// block, a wave each (fwd_tail_rows), in front of all others; as many blocks as a multiple of 8, so that the others stay on the
// XCD of their slice.  Work group `lin` and wave -> slice; one past the last means none.
FMHA_HOST_DEVICE int fmha_tail_blocks(int slices, int per) { return ((slices + per - 1) / per + 7) & ~7; }
FMHA_HOST_DEVICE int fmha_tail_slice(int lin, int wave, int tails, int per) {
  return per * ((lin & 7) * (tails >> 3) + (lin >> 3)) + wave;  // an XCD has slices next to each other here too
}

// Whether they do: 0, or how many to a block.  Blocks of the same length are done in layers of one to a CU, and it pays where
// there are fewer of those.  Two to a block where that gives as few as four does, since four streams of K and V are slow beside
// another block.  us of the forward with a block for each, two and four to a block, N x slices (layers):
// D = 64.  129 x 230 (2, 2, 2) 7.8, 8.0, 8.3; 129 x 300 (3, 2, 2) 11.5, 8.7, 8.7; 129 x 400 (4, 3, 2) 13.9, 11.8, 9.5; 129 x
// 512 (4, 3, 3) 16.4, 12.1, 12.8; 129 x 4000 (32, 24, 20) 99.0, 80.2, 77.8; 257 x 100 (2, 1, 1) 9.6, 7.7, 7.8; 257 x 400 (5, 4,
// 4) 24.9, 22.1, 21.8; 520 x 110 (3, 2, 2) 21.8, 17.1, 18.1; 520 x 120 (3, 3, 2) 22.0, 22.1, 18.4; 520 x 150 (3, 3, 3) 24.0,
// 24.4, 23.4; 660 x 90 (3, 2, 2) 24.9, 19.8, 20.7; 1031 x 56 (2, 2, 2) 26.5, 27.2, 27.9; 1031 x 60 (3, 2, 2) 31.8, 27.9, 28.5;
// 1031 x 230 (9, 8, 8) 98.5, 94.6, 92.4; 2070 x 31 (3, 2, 2) 54.5, 48.8, 49.7; 2070 x 200 (14, 13, 13) 276, 275, 268.
// D = 128.  129 x 230 (2, 2, 2) 13.7, 11.9, 13.7; 129 x 300 (3, 2, 2) 19.6, 13.2, 14.8; 257 x 200 (3, 2, 2) 23.9, 20.2, 21.8;
// 257 x 700 (9, 7, 7) 67.2, 60.4, 57.2; 520 x 56 (2, 1, 1) 20.9, 17.9, 18.8; 520 x 64 (2, 2, 2) 21.9, 23.1, 24.4; 520 x 600
// (12, 11, 10) 138, 136, 130; 1031 x 56 (2, 2, 2) 41.9, 44.2, 46.0; 1031 x 60 (3, 2, 2) 50.1, 46.0, 48.0; 1031 x 120 (5, 4, 4)
// 87.9, 82.7, 81.0; 1300 x 48 (3, 2, 2) 58.2, 53.8, 56.8; 2070 x 31 (3, 2, 2) 88.6, 81.8, 84.2.
// Not past three rounds of longer ones at D = 128: 1031 x 200 (8, 7, 7) 146, 150, 150; 2070 x 230 (16, 15, 15) 550, 579, 539.
// Nor from two layers to one where it is the wave on its own that takes the time: D = 64 660 x 45 15.6, 13.8, 15.4; 1031 x 30
// 20.4, 20.6, 21.7; 1300 x 24 23.8, 24.9, 25.9; and with four to a block 900 x 34 18.7, 21.7, 19.5.  D = 128 1031 x 30 31.8,
// 29.1, 31.7; 900 x 34 28.8, 32.8, 28.8.
// Under causal masking these rows have more keys than any others, and go first anyhow.  Up to 160 rows, where that makes two
// kinds of block alike, by the layers too (D = 64 129 x 300 40, 129 x 400 13 and 57 % faster; D = 128 150 x 300 29 and 15, 150
// x 256 (2, 2, 2) 7 and 11 slower).  Longer ones: a launch must last longer than a wave for itself takes, and the fewer blocks
// of a slice the more there is to gain; with a block for each and four to a block: D = 64 257 x 230 14.0, 12.3; 400 x 200 17.8,
// 15.8; 520 x 180 1 % better, 520 x 512 5 %, 520 x 100 11 % worse; D = 128 257 x 219 19.5, 16.0; 288 x 376 29.8, 26.8; 385 x
// 216 27.1, 24.9; 410 x 181 22.3, 22.3; 530 x 170 29.4, 28.1; 520 x 100 17 % worse.  Past 576 rows 1 to 2 % in the mean, with
// losses among them; and hardly anything, or less, where the blocks are just past full layers: D = 128 410 x 264 (5) 31.8,
// 33.2; 257 x 257 (4) 21.2, 21.9; D = 64 410 x 257 (5) 20.3, 20.6.
// And the more rounds (in brackets) the less: D = 128 257 x 624 (7.3) 42.3, 40.0; 288 x 625 (7.3) 43.5, 42.2; 257 x 641 (7.5)
// 43.5, 43.0; 288 x 641 (7.5) 44.8, 46.0; 257 x 737 (8.6) 48.6, 49.0; 288 x 737 (8.6) 50.1, 52.2; 385 x 441 (6.9) 46.4, 45.5;
// 400 x 417 (6.5) 45.6, 46.1; 400 x 481 (7.5) 51.3, 52.0; 400 x 537 (8.4) 56.3, 56.8; 416 x 249 (3.9) 30.5, 29.0; 416 x 276
// (4.3) 32.1, 32.7; 416 x 353 (5.5) 39.7, 41.4; 416 x 417 (6.5) 45.6, 46.6; 513 x 301 (5.9) 47.0, 45.9; 544 x 289 (5.6) 46.2,
// 46.5; 513 x 324 (6.3) 48.6, 49.8; 544 x 385 (7.5) 58.2, 61.5; 513 x 455 (8.9) 67.2, 69.2; D = 64 416 x 489 (7.6) 33.7, 32.2.
FMHA_HOST_DEVICE int fmha_tails_per_block(int d, int n, int slices, int cus, bool causal) {
  if (n <= 128 || (n - 1) % 128 >= 32) return 0;
  const long full = (long)slices * ((n - 1) / 128);
  const long now = (full + slices + cus - 1) / cus, two = (full + fmha_tail_blocks(slices, 2) + cus - 1) / cus,
             four = (full + fmha_tail_blocks(slices, 4) + cus - 1) / cus;
  if (causal && n > 160) {
    const long blocks = full + slices, left = blocks % cus;
    const int most = n <= 288 ? 15 : n <= 400 ? 14 : n <= 512 ? 8 : 12;  // half rounds of blocks
    if (d == 128 && 2 * blocks >= (long)most * cus) return 0;
    return n <= 576 && 480 * blocks >= (900L + n) * cus && 16 * left >= (d == 64 ? 1 : 5) * cus ? 4 : 0;
  }
  if (n > 768 && ((d == 128 && now > 6) || (now == 2 && (d == 64 || two == 2)))) return 0;
  return two < now && two <= four ? 2 : four < now ? 4 : 0;
}

// A launch of two passes with `nb` blocks each per slice: the blocks of both in turn, ordered as one pass's are (heaviest of
// both first, or the short last ones of both at the end).
// `run`, last_level: as in fmha_ordered_block, of 2 * nb blocks, the last two short ones.
template <typename Int>
FMHA_HOST_DEVICE void fmha_two_pass_ordered_block(int lin, int slices, const Int& run, const Int& last_level, bool heavy_first,
                                                  bool short_last, int& slice, int& blk, bool& second_pass) {
  int v;
  if (heavy_first || !short_last || lin < slices * run) {
    fmha_ordered_block(lin, slices, run, last_level, heavy_first, false, slice, v);
  } else {
    slice = (lin - slices * run) >> 1;
    v = run + ((lin - slices * run) & 1);
  }
  blk = v >> 1;
  second_pass = v & 1;
}
FMHA_HOST_DEVICE void fmha_two_pass_block(int lin, int slices, int nb, bool heavy_first, bool short_last, int& slice, int& blk,
                                          bool& second_pass) {
  const int run = 2 * fmha_blocks_in_order(nb, heavy_first, short_last);
  fmha_two_pass_ordered_block(lin, slices, run, fmha_last_level(slices), heavy_first, run < 2 * nb, slice, blk, second_pass);
}

// A launch of all blocks of the dK/dV pass and then all of the dQ pass over the dS that it stores, nb each per slice, either in
// the order of a launch of its own (the short last blocks of sequences without a mask in their places: what comes last are the
// dQ blocks, and they wait for whole slices).  The second part begins at a multiple of 8, so that a slice stays on its XCD; the
// up to 7 work groups before that have no block.
FMHA_HOST_DEVICE int fmha_ds_launch_blocks(int slices, int nb) { return ((slices * nb + 7) & ~7) + slices * nb; }
template <typename Int>
FMHA_HOST_DEVICE bool fmha_ds_launch_ordered_block(int lin, int slices, const Int& nb, const Int& last_level, bool heavy_first,
                                                   int& slice, int& blk, bool& second_pass) {
  const int blocks = slices * nb, second = (blocks + 7) & ~7;
  second_pass = lin >= second;
  if (second_pass) lin -= second;
  if (lin >= blocks) return false;
  fmha_ordered_block(lin, slices, nb, last_level, heavy_first, false, slice, blk);
  return true;
}
FMHA_HOST_DEVICE bool fmha_ds_launch_block(int lin, int slices, int nb, bool heavy_first, int& slice, int& blk,
                                           bool& second_pass) {
  return fmha_ds_launch_ordered_block(lin, slices, nb, fmha_last_level(slices), heavy_first, slice, blk, second_pass);
}

// What the kernels take of a launch whose blocks are numbered in one of the orders above.
// us of forward and backward kernels with the divisions of ints, then with these, in graphs of 20 calls, N x slices: D = 64
// 77 x 8 causal 5.85, 5.76 and 7.02, 6.86; 300 x 80 causal 7.74, 7.65 and 13.5, 13.4; backward 256 x 256 23.1, 22.8; D = 128 200 x 48
// causal 9.59, 9.45 and 15.1, 14.8; 2048 x 80 causal 95.5, 95.7 and 304, 297; 1031 x 60 43.2 both and 115.9, 114.6.
struct FmhaOrder {
  FmhaDivisor run, last_level;
  int slices;
  bool short_last;  // the short last blocks come at the end
  FmhaOrder() = default;
  FMHA_HOST FmhaOrder(int slices_, int blocks_per_slice, bool heavy_first, bool short_last_, int passes = 1)
      : run(passes * fmha_blocks_in_order(blocks_per_slice, heavy_first, short_last_)), last_level(fmha_last_level(slices_)),
        slices(slices_), short_last((int)run < passes * blocks_per_slice) {}
};

// How long a dQ block of that launch waits for the dS of its slice before it forms S and dP itself, in ticks of 10 ns.  Blocks
// are handed out in order inside an XCD only, and a slice that no XCD has for itself (slices % 8) has blocks on several.  With
// launches on more than one stream, dQ blocks of one that wait can so hold all CUs that dK/dV blocks of another need, and the
// other way round.  So a block waits long only for dK/dV blocks that have all started: these wait for nobody and take 16 ns a
// row of the slice.  For others it waits about as long as it takes to do without them.
FMHA_HOST_DEVICE unsigned fmha_ds_wait_ticks(int n, bool started) { return (500u + 2u * (unsigned)n) * (started ? 32u : 1u); }

// Whether such a launch takes the place of the two passes one after the other.  It gains where the last round of one of them is
// far from full, and with few rounds, and a launch where these are short; it loses where a dQ block of 128 queries is much
// slower than the one of 256 that the dQ pass alone takes then (half of the copies of K), which long sequences feel.  us of the
// backward, passes apart and in one launch, N x slices (rounds of blocks of 128 rows):
// Up to 768 rows.  64 x 520 (2.0) 40.3, 30.4; 64 x 1200 (4.7) 59.5, 59.4; 100 x 300 (1.2) 44.2, 34.9; 100 x 3000 (11.7) 226,
// 235; 128 x 600 63.1, 50.9; 128 x 2000 (7.8) 177, 174; 200 x 200 46.0, 37.3; 256 x 256 (2) 52.5, 51.5; 300 x 86 (1.0) 42.3,
// 32.5; 384 x 400 (4.7) 159, 144; 512 x 64 (1) 38.2, 35.7; 512 x 100 63.4, 54.9; 512 x 192 (3) 107, 103; 512 x 256 (4) 140,
// 141; 512 x 600 (9.4) 346, 345; 640 x 128 (2.5) 112, 97; 640 x 300 (5.9) 251, 243.  Causal: 64 x 600 43.5, 33.9; 64 x 2000
// (7.8) 98.0, 98.2; 128 x 1200 (4.7) 117, 99; 200 x 400 69.9, 58.3; 200 x 1000 (7.8) 153, 157; 256 x 300 62.5, 50.7; 256 x 1000
// 191, 184; 512 x 80 42.4, 37.6; 512 x 192 (3) 86.7, 78.2; 512 x 400 (6.3) 176, 171; 640 x 200 (3.9) 123, 114.
// Longer, without a mask.  One round or less: 1024 x 32 59.2, 55.5; 1280 x 20 59.6, 57.6; 2048 x 16 97.0, 95.9; 4096 x 8 185,
// 193.  777 x 40 (1.1) 69.4, 58.2; 777 x 100 (2.7) 136, 125; 1024 x 48 (1.5) 96.2, 86.0; 1024 x 64 (2) 107, 106; 1024 x 96 (3)
// 165, 167; 1031 x 60 (2.1) 129, 114; 1500 x 24 (1.1) 123, 105; 1500 x 48 (2.3) 204, 177; 1500 x 64 (3) 232, 234; 1500 x 100
// (4.7) 374, 375; 2048 x 20 (1.3) 158, 135; 2048 x 28 (1.8) 189, 186; 2048 x 56 (3.5) 368, 353; 2048 x 64 (4) 397, 404; 2048 x
// 130 (8.1) 872, 839; 2048 x 170 (10.6) 1089, 1100; 3000 x 12 (1.1) 230, 195; 3000 x 50 (4.7) 664, 677; 4096 x 10 (1.3) 309,
// 263; 4096 x 20 (2.5) 506, 482; 4096 x 32 (4) 710, 739; 4096 x 42 (5.3) 1002, 992; 4096 x 52 (6.5) 1230, 1239; 6000 x 6 (1.1)
// 435, 435; 6000 x 8 (1.5) 470, 473; 6000 x 12 (2.2) 705, 618; 8192 x 5 (1.3) 574, 582; 8192 x 9 (2.3) 909, 828; 8192 x 17
// (4.3) 1606, 1540; 16384 x 3 1189, 1211.
// Longer, causal.  777 x 64 (1.8) 58.0, 54.8; 777 x 300 (8.2) 267, 262; 1024 x 40 54.6, 50.4; 1024 x 128 (4) 144, 146; 1024 x
// 150 190, 176; 1024 x 220 (6.9) 276, 264; 1280 x 100 (3.9) 176, 170; 1500 x 48 (2.3) 118, 108; 1500 x 80 (3.8) 189, 181; 2048
// x 20 85.3, 81.0; 2048 x 56 (3.5) 213, 208; 2048 x 64 (4) 232, 237; 2048 x 80 (5) 296, 299; 4096 x 9 (1.1) 149, 140; 4096 x 11
// (1.4) 159, 153; 4096 x 12 (1.5) 169, 171; 4096 x 16 (2) 207, 210; 8192 x 6 323, 324; 8192 x 12 (3) 586, 594; 16384 x 16 (8)
// 2820, 2919.
// Past six rounds the figures above leave out what the one launch pays for dS past the L2s when others follow; us of forward
// and backward as calls, in two launches and in one, no mask: 260 x 631 (7.4) 241, 230; 384 x 631 (7.4) 316, 313; 400 x 473
// (7.4) 295, 294; 768 x 315 (7.4) 462, 456; 777 x 230 (6.3) 383, 377; 777 x 303 (8.3) 520, 512; 1000 x 265 (8.3) 666, 634; 1024
// x 265 (8.3) 656, 638; 1500 x 110 (5.2) 589, 572; 1500 x 155 (7.3) 814, 800; 2048 x 84 (5.3) 757, 741; 2048 x 100 (6.3) 912,
// 915; 2048 x 114 (7.1) 1017, 1020; 2048 x 130 (8.1) 1178, 1191; 4096 x 42 (5.3) 1390, 1373.  Causal: 400 x 473 (7.4) 223, 223;
// 700 x 268 (6.3) 245, 246; 768 x 315 (7.4) 322, 317; 777 x 193 (5.3) 214, 210; 777 x 239 (6.5) 268, 268; 896 x 193 (5.3) 247,
// 244; 896 x 239 (6.5) 315, 309; 900 x 129 (4.0) 184, 182; 1024 x 129 (4.0) 207, 203; but 900 x 145 (4.5) 201, 202; 900 x 169
// (5.3) 231, 235; 960 x 161 (5.0) 231, 232; 960 x 185 (5.8) 266, 269; 1024 x 185 (5.8) 294, 296; 1024 x 220 (6.9) 353, 350.
FMHA_HOST_DEVICE bool fmha_ds_in_one_launch(int slices, int n, int cus, bool causal) {
  const long blocks = (long)slices * ((n + 127) / 128), left = blocks % cus;
  if (n <= 768) return 2 * blocks <= 15L * cus;
  if (causal) {
    if (n <= 1024) return 8 * blocks <= (n <= 896 ? 56L : 33L) * cus;
    return n <= 2048 ? blocks < 4L * cus : n <= 4096 && 2 * blocks < 3L * cus;
  }
  if (blocks <= cus) return n <= 2048;
  if (left == 0) return false;
  if (n <= 1024) return 4 * left <= 3L * cus && blocks <= 9L * cus;
  if (n <= 4096) return 2 * left <= cus && blocks <= (n <= 1536 ? 8L : 6L) * cus;
  return n <= 8192 && 4 * left <= cus && blocks > 2L * cus && blocks < 5L * cus;
}

// Whether the backward takes a work group for each slice (fmha_bwd_slice_kernel, one to a CU), before all of the below.  It
// forms S and dP once, as the D = 128 passes over dS do, but needs no room for dS, makes the statistics and is one launch; and
// it reads Q, K, V and dO once.  It loses where slices leave CUs idle that blocks of 128 rows would fill: with few slices, and
// with a last round that is far from full, the more so the longer a round is and under causal masking, where half of the blocks
// of a slice are light, which the other launches pair with heavy ones.  At D = 64 up to 128 rows half of its waves have no
// keys, and blocks of 128 rows, two to a CU, are ahead (64 x 256, 128 x 256 and 128 x 1024 lose 6, 2 and 15 %).
// The lines are where the two were as fast when a work group per slice took 4 to 13 % longer than now, and were left there.  The
// times are of the kernels as they are, in graphs of 20 calls, each side behind itself, mean of two cards, which differ by up to 5 %
// in what one side takes of the other.  So some entries that the rule leaves to the passes are slower there, by up to 18 % (D = 64,
// 512 x 1030).
// us of the kernels of the backward, without it and with it, N x slices:
// D = 128, without a mask.  One round: 40 x 128 7.1, 8.9; 40 x 160 12.2, 9.1; 200 x 128 25.3, 25.2; 256 x 136 41.0, 27.5; 256 x
// 256 50.7, 35.8.  Two: 17 x 264 17.1, 12.3; 100 x 264 27.3, 26.3; 160 x 288 41.6, 43.6; 160 x 320 45.6, 43.4; 256 x 288 56.5,
// 56.9; 256 x 320 62.4, 58.0; 256 x 512 97.1, 70.6.  More: 33 x 514 23.8, 23.5; 50 x 528 27.4, 27.0; 100 x 528 41.0, 41.6; 100 x
// 640 47.0, 42.1; 100 x 800 58.2, 56.4; 100 x 1030 70.1, 70.5; 100 x 1600 116, 108; 256 x 528 107, 94.0; 256 x 1024 204, 158.
// D = 128, causal.  160 x 128 19.4, 17.0 but 200 x 128 23.3, 22.1 and 100 x 128 slower; 256 x 160 33.8, 26.1; 256 x 256 42.0,
// 30.9; 160 x 288 35.8, 32.7; 256 x 288 46.9, 50.2; 256 x 336 53.3, 51.4; 256 x 352 55.9, 52.4; 256 x 512 83.1, 60.3; 100 x 514
// 39.4, 39.5; 100 x 640 46.8, 40.9; 256 x 528 87.3, 82.2.
// D = 64, without a mask.  256 x 128 14.4, 17.5; 145 x 144 15.2, 12.8; 256 x 144 19.8, 17.9; 300 x 168 30.2, 31.8; 300 x 192
// 34.2, 31.6; 512 x 192 61.1, 52.7; 512 x 256 80.5, 59.6; 300 x 352 61.1, 60.1; 300 x 384 62.3, 61.5; 300 x 400 64.3, 61.9; 512 x
// 384 115, 105; 512 x 448 134, 111; 300 x 560 86.3, 89.4; 300 x 600 93.0, 89.7; 512 x 560 168, 161; 512 x 620 185, 166; 300 x 770
// 116, 118; 300 x 900 131, 124; 300 x 1030 154, 155; 512 x 1030 328, 277; 512 x 1300 411, 340.
// D = 64, causal.  129 x 160 12.3, 11.5; 129 x 168 12.5, 11.5; 160 x 256 17.4, 13.4; 145 x 416 25.4, 24.0; 145 x 448 26.8, 24.6;
// 145 x 600 34.0, 34.8; 180 x 208 15.6, 14.4; 200 x 230 18.9, 16.8; 256 x 240 21.3, 20.1; 300 x 208 25.8, 25.3; 300 x 230 28.6,
// 25.4; 300 x 480 53.8, 50.1; 300 x 496 59.7, 50.5; 512 x 208 46.9, 42.8; 512 x 230 50.8, 43.6; 512 x 256 58.4, 45.3; 512 x 432
// 91.4, 84.9; 512 x 448 95.3, 85.7; 512 x 512 107, 89.2; 512 x 640 137, 134; 512 x 720 160, 143; 512 x 800 185, 179; 512 x 900
// 212, 183; 512 x 1030 238, 220; 300 x 1030 118, 121.
// D = 64 without a mask, 385 to 512 rows, one round: the line is at the fewest slices that were timed, not where the passes are
// as fast.  A round takes as long with fewer: 512 x 176 57.9, 50.5.
// Causal, D = 128, a second round of slices just past 96 rows (four tiles of 32 queries instead of three), us of forward and
// backward, without it and with it: 97 x 257 34.4, 34.5; 97 x 266 34.7, 36.0; 97 x 296 35.9, 36.3; 97 x 320 36.6, 36.0; 105 x 266
// 35.8, 36.3; 105 x 306 37.3, 36.3; 112 x 266 36.9, 36.5; 112 x 306 38.3, 36.6; 116 x 266 37.5, 36.8; 128 x 266 38.7, 37.4; and
// 96 x 257 33.1, 31.4.
// D = 64 without a mask, 161 to 176 rows, us of forward and backward, without it and with it: 161 x 598 64.3, 62.6; 161 x 612
// 64.1, 62.3; 161 x 652 68.7, 65.5; 176 x 612 65.9, 64.5; 176 x 652 70.5, 66.5; 161 x 1812 166, 167; 161 x 1892 171, 169; 161 x
// 1932 178, 174; 176 x 1812 171, 173; 176 x 1932 186, 180; 161 x 2068 192, 191; 176 x 2068 204, 198.
// Causal, D = 64, 161 to 200 rows, us of forward and backward, without it and with it: 161 x 224 23.0, 23.9; 161 x 256 25.2,
// 24.8; 170 x 236 24.4, 24.3; 180 x 224 23.5, 24.6; 180 x 244 25.4, 24.9; 192 x 224 23.6, 24.8; 192 x 236 24.7, 24.7; 192 x 250
// 25.5, 25.1; 193 x 224 27.3, 27.8; 193 x 250 28.7, 28.8; 200 x 230 27.9, 27.8; 200 x 240 28.1, 28.1; 200 x 256 30.3, 28.1.
// From 257 to 384 rows at D = 64 the line depends on the last tile of 64 rows too, of which the other launches do all even if
// only half of it has rows (257 to 288 and 321 to 352 rows).  us of forward and backward, without it and with it, N x slices:
// last tile whole, no mask: 290 x 448 98.4, 91.1; 384 x 448 119, 105; 290 x 704 142, 136; 304 x 960 193, 184; 384 x 1216 313,
// 279; 290 x 1216 237, 232; 290 x 1440 284, 281; 320 x 1440 299, 279; 289 x 1576 318, 316; 304 x 1704 346, 333; but 384 x 385
// 101, 97.1; 290 x 598 123, 124; 290 x 833 163, 166; 320 x 1076 210, 212; 290 x 1352 260, 269; 304 x 1544 318, 318.
// Causal: 320 x 248 44.5, 41.1; 384 x 248 52.1, 48.8; 384 x 496 97.2, 90.1; 320 x 1264 203, 190; 289 x 1520 242, 223; but 320 x
// 224 40.3, 39.0; 384 x 224 47.5, 46.4; 384 x 752 139, 134; 320 x 1014 154, 148.
// Last tile half empty, no mask: 264 x 608 117, 111; 264 x 840 152, 149; 352 x 400 103, 93.4; 352 x 840 198, 185; 352 x 1080 254,
// 241; 264 x 1336 234, 227; 352 x 1320 324, 298.  Causal: 264 x 232 39.1, 35.0; 352 x 224 45.5, 42.6; 264 x 752 107, 94.4; 352 x
// 1008 181, 166.
FMHA_HOST_DEVICE bool fmha_backward_by_slice(int d, int n, int slices, int cus, bool causal) {
  if (n > 32768 / d) return false;  // LDS and registers hold no more keys
  const long rounds = ((long)slices + cus - 1) / cus, last = slices - (rounds - 1) * cus;
  if (d == 128) {
    if (rounds == 1) return 2 * last > cus;
    if (n <= 64) return true;
    if (rounds == 2 && causal && n > 96 && n <= 112) return 5 * last >= cus;
    if (n <= 128) return rounds == 2 || rounds > 6 || 2 * last >= cus;
    return rounds > 2 || (causal && n > 160 ? 3 : 4) * last >= cus;
  }
  if (n <= 128) return false;
  const bool whole_tiles = (n - 1) % 64 >= 32;
  if (!causal) {
    if (rounds == 1) return n <= 256 ? 2 * last > cus : 4 * last >= 3L * cus;
    if (n > 256 && n <= 384 && whole_tiles) return 8 * last >= (rounds < 6 ? 6L : rounds == 6 ? 5L : 1L) * cus;
    if (n > 160 && n <= 176 && (rounds == 3 || rounds == 8 || rounds == 9)) return 5 * last >= 2L * cus;
    return rounds > 5 || rounds * last > cus;
  }
  if (n <= 160) return rounds == 1 ? 3 * last >= 2L * cus : rounds == 2 && 4 * last >= 3L * cus;
  if (n <= 256) return n <= 200 && rounds == 1 && 16 * last >= (n <= 184 ? 14L : 16L) * cus;
  if (n <= 384 && whole_tiles) return rounds != 3 && rounds != 4 && 16 * last >= 15L * cus;
  if (n <= 384) return 16 * last >= (rounds == 1 ? 14L : 15L) * cus;
  return rounds > 4 || 8 * last >= (rounds == 1 ? 7L : 6L) * cus;
}

// Whether the backward does both passes, `blocks` blocks of 128 rows each, in one launch of 2 * blocks.  With fewer blocks
// than places (D = 64: two to a CU, D = 128: one) the passes one after the other leave most of the chip idle; with a few more,
// each has a nearly empty last round of its own.  Where the one launch takes as many rounds as the two passes together it
// saves launches, and pays for the statistics, which the D = 64 dQ pass makes on the side when it goes first, or, at D = 128,
// for forming S and dP twice; most where the last tile is not whole.  The launches it saves are one at D = 64, two and the
// room for dS at D = 128: 4 and 7 us of the host, and a program that calls these functions from Python waits for the host
// unless forward and backward have 40 us of kernels or, more often, 70.  us of the two through autograd, one launch and apart:
// D = 128 N = 64 x 256 slices 71, 79 (kernels of the backward 16.9, 15.5); 100 x 256 73, 79; 40 x 448 73, 79; 100 x 448 75, 80
// (kernels 44.4, 39.6); 180 x 192 73, 80; causal 40 x 480 73, 79; D = 64 64 x 512 72, 77; 80 x 448 73, 76.  So short launches
// go in one also where their kernels lose by it, up to 3 us, and at D = 128 without a mask from 65 to 127 rows past one and a
// half blocks per CU 4 to 8; the lines lie where a call waits for its kernels, or where they lose more.
// us of the kernels one after the other, and of one launch with the statistics made by the blocks or, behind "+", by a kernel
// of their own first (fmha_blocks_make_stats), N x slices (blocks per CU), on both sides of the lines:
// D = 64, without a mask, up to 256 rows.  64 x 512 (2) 14.0, 15.0; 80 x 448 (1.75) 17.7, 18.7; 120 x 512 22.0, 23.9; 120 x
// 538 (2.1) 28.9, 24.8; 128 x 512 23.0, 20.6; 204 x 256 30.7, 29.0; 255 x 256 equal.  Many blocks: 24 x 3840 (15) 58.8, 58.5;
// 24 x 5120 75.4, 76.7; 40 x 3840 64.7, 63.3; 40 x 4096 (16) 68.5, 71.6; 64 x 2048 (8) 44.3, 42.9; 64 x 2432 53.0, 55.1; 64 x
// 3584 69.4, 74.5; 80 x 2048 56.4, 57.6; 80 x 2560 68.5, 71.9; 128 x 2048 74.4, 69.3; 256 x 640 (5) 64.6, 60.4; 256 x 768
// 73.3, 77.0.
// Longer: 512 x 32 22.5, 14.9; 512 x 96 (1.5) 37.3, 33.7; 512 x 112 39.3, 40.9; 512 x 128 (2) 42.0, 44.2; 512 x 136 54.8,
// 50.8; 512 x 160 (2.5) 55.9, 53.5; 512 x 176 57.5, 60.8; 512 x 208 (3.25) 70.4, 70.3.  4096 x 4 (0.5) 118, + 75.5; 2048 x 24
// (1.5) 110, + 103; 2048 x 28 118, + 126; 2048 x 32 (2) 128, + 134; 2048 x 40 (2.5) 173, + 168; 2048 x 44 179, + 190; 4096 x
// 26 (3.25) 440, + 424; 4096 x 28 449, + 438; 4096 x 30 462, + 484; 4096 x 36 (4.5) 554, + 561.
// D = 64, causal.  1 x 4096 (16) 57.2, 56.9; 1 x 5120 69.9, 70.3; 25 x 5120 (20) 82.7, 81.4; 140 x 1024 (8) 61.7, 56.2; 450 x
// 320 (5) 69.5, 66.3; 450 x 352 72.5, 73.3; 512 x 512 (8) 110, 117; 777 x 144 (3.95) 70.4, 66.3; 1024 x 32 37.9, 27.3; 1024 x
// 128 (4) 86.3, 85.7; 2048 x 32 (2) 79.9, + 74.3; 2048 x 60 136, + 135; 2048 x 64 (4) 141, + 145; 8192 x 8 (2) 283, + 256;
// 8192 x 15 464, + 459; 8192 x 32 946, + 963.
// D = 128, without a mask.  33 x 128 (0.5) 14.1, 7.8; 33 x 256 (1) 14.7, 13.3; 64 x 256 15.5, 16.9; 64 x 264 23.9, 22.5; 64 x
// 397 (1.55) 27.2, 30.4; 48 x 486 (1.9) 25.3, 28.4; 64 x 512 (2) 29.2, 32.1; 64 x 537 41.4, 37.2; 110 x 128 18.7, 13.2; 120 x
// 140 (0.55) 19.8, 23.1; 110 x 256 24.1, 26.1; 110 x 384 (1.5) 38.4, 38.1; 80 x 396 33.9, 40.2; 110 x 410 39.7, 46.1; 120 x
// 512 45.5, 50.8.  128 x 128 19.0, 12.2; 128 x 141 19.6, 20.8; 128 x 256 24.8, 24.2; 128 x 384 40.3, 34.5; 128 x 410 41.5,
// 43.7; 128 x 512 47.0, 44.8; 128 x 537 61.2, 53.5.  140 x 64 (0.5) 19.6, 12.8; 140 x 68 20.1, 20.5; 140 x 128 (1) 23.7, 24.7;
// 140 x 141 33.2, 33.9; 140 x 192 (1.5) 37.0, 36.3; 200 x 64 22.6, 16.4; 200 x 68 22.9, 27.5; 200 x 141 41.0, 42.5; 230 x 192
// 47.5, 48.5; 200 x 198 (1.55) 46.4, 56.9; 256 x 132 43.8, 43.0; 256 x 192 46.7, 45.4; 256 x 205 48.5, 57.3.  350 x 38 (0.45)
// 26.9, 20.1; 350 x 43 27.2, 34.6; 1200 x 11 (0.43) 49.6, + 40.1; 1200 x 13 49.4, + 67.8; 2048 x 8 (0.5) 75.4, + 64.5; 4096 x
// 4 (0.5) 131, + 122; 4096 x 5 145, + 209.
// D = 128, causal.  24 x 384 (1.5) 23.1, 18.0; 24 x 410 23.3, 22.8; 40 x 486 (1.9) 24.1, 25.8; 64 x 512 (2) 30.7, 28.2; 64 x
// 537 43.3, 34.3; 110 x 410 40.0, 40.2; 110 x 512 45.5, 43.3; 129 x 128 (1) 21.7, 21.5; 129 x 192 33.0, 30.5; 200 x 192 (1.5)
// 41.5, 35.9; 200 x 218 42.2, 43.3; 512 x 64 (1) 37.7, + 34.2; 512 x 68 41.5, + 43.2; 777 x 33 (0.9) 42.0, + 37.8; 2048 x 16
// (1) 84.9, + 76.0; 2048 x 18 91.6, + 89.2; 2048 x 20 91.1, + 98.1; 4096 x 8 (1) 153, + 133; 4096 x 10 159, + 169; 8192 x 5
// 315, + 318.
// room: whether the workspace holds dS.  If not, the D = 128 passes one after the other form S and dP twice as well, and
// without a mask a round saved counts at any length: 1031 x 42 (1.5) 121, 106; 4096 x 9 (1.1) 388, 318; 16384 x 3 1554, 1326.
// Under causal masking the lines are those with room, though the one launch is ahead past them: 1024 x 48 (1.5) 76.8, 72.1;
// 1024 x 64 (2) equal; 2048 x 24 117, 108.
FMHA_HOST_DEVICE bool fmha_passes_at_once(int d, long blocks, int n, int cus, bool causal, bool room = true) {
  if (d == 128) {
    if (blocks > 2L * cus) return false;
    if (n <= 128) return true;
    if (causal) return 2 * blocks <= (n <= 256 ? 3L : 2L) * cus;
    const bool three_rounds_for_four = blocks > cus && 2 * blocks <= 3L * cus;
    return 2 * blocks <= cus || (three_rounds_for_four && (n <= 256 || !room));
  }
  const long places = 2L * cus;
  if (causal) return n <= 512 ? blocks <= 10 * places && blocks * n <= places * (2L * n + 256) : blocks < 2 * places;
  if (n <= 256) return 2 * blocks < (n <= 60 ? 15 : 10) * places && blocks * n <= places * (n + 384L);
  const long left = 2 * blocks % places;
  return 4 * blocks <= 3 * places || (blocks > places && blocks < 2 * places && left > 0 && 2 * left <= places);
}

// Whether the blocks of such a launch make the row statistics themselves, which adds a tenth and more to the tiles of the
// dK/dV blocks, or a kernel before it does, which takes 2 to 5 us and more where there are many rows.  Figures as above,
// blocks, then kernel.  D = 64: 256 x 64 10.4, 12.1; 512 x 32 14.9, 15.9; 512 x 160 53.5, 53.2; 1024 x 16 24.9, 24.4; 1024 x 48
// 59.8, 56.9; 4096 x 4 85.3, 75.5; causal 512 x 64 17.8, 18.9; 1024 x 16 24.1, 23.5; 1024 x 64 43.4, 45.2; 1024 x 104 70.1, 73.5;
// 2048 x 12 44.5, 41.0; 8192 x 4 172, 155.  D = 128: 128 x 32 9.7, 10.9; 256 x 16 13.4, 13.8; 256 x 64 16.0, 17.4; 512 x 8 21.0,
// 19.2; 512 x 32 24.1, 24.0; 1024 x 8 36.5, 30.9; causal 256 x 64 15.3, 16.5; 512 x 8 21.3, 20.0; 512 x 40 24.6, 25.0; 1024 x 16
// 37.0, 32.4.
FMHA_HOST_DEVICE bool fmha_blocks_make_stats(int d, int n, bool causal) {
  return n <= (d == 128 ? 384 : causal ? 1024 : 512);
}

// Whether the D = 128 passes over dS are told that it is used once.  Without that dS stays in the 256 MiB Infinity Cache
// between the two: better where it fits together with the six tensors the passes touch, and is not small.  Small is less than
// 16 MiB without a mask up to 384 rows, 8 MiB (of half the square) under causal masking and 10 MiB else.  Fewer blocks than
// those of the figures go in one launch that stores no dS, unless the passes are called one by one, as the ones with "*" are.
// us of the backward without and with the hint, N x slices (MiB of dS; with the tensors):
// Lower line: 66 x 230 * (7; 29) 20.3, 19.0; 110 x 256 * (8; 49) 24.7, 24.4; 77 x 430 * (13; 62) 36.5, 35.9; 140 x 79 (10; 26)
// 20.7, 20.3; 140 x 120 (15; 40) 23.2, 22.3; 200 x 110 (14; 46) 26.8, 26.5; 256 x 100 (13; 50) 27.0, 26.8; 256 x 128 (16; 64)
// 30.4, 30.7; 257 x 46 (13; 30) 25.2, 24.2; 384 x 46 (13; 39) 28.2, 27.9; 384 x 64 (18; 54) 29.9, 29.9; 384 x 85 (24; 72)
// 33.3, 34.0; 200 x 135 (17; 56) 42.1, 42.2; 110 x 520 (16; 100) 57.6, 58.5; 128 x 520 (16; 114) 61.3, 62.6; 350 x 86 (24; 68)
// 51.8, 53.6; causal 33 x 500 * (8; 32) 24.0, 23.5; 50 x 500 * (8; 44) 26.7, 26.5; 64 x 530 (8; 58) 43.4, 43.4; 128 x 513 (8;
// 104) 59.3, 61.0; 128 x 600 (9; 122) 64.3, 65.3; 512 x 75 (19; 75) 45.0, 47.7.  Forward and backward: 512 x 16 * (8; 20)
// 40.8, 39.8; 1024 x 5 * (10; 18) 59.8, 61.8.
// Upper line, forward and backward: 1031 x 60 (152; 243) 203, 207; 4096 x 11 causal (176; 242) 240, 254; 512 x 224 (112; 280)
// 185, 179; 1024 x 88 (176; 308) 237, 227; 4096 x 16 causal (256; 352) 305, 300; 4096 x 64 causal (1024; 1408) 1217, 1161.
FMHA_HOST_DEVICE bool fmha_ds_used_once(unsigned long ds_bytes, unsigned long touched, int n, bool causal) {
  const unsigned long small = causal ? 8 : n <= 384 ? 16 : 10;  // MiB
  return ds_bytes < (small << 20) || touched > (256ul << 20);
}

// Row statistics: blocks of consecutive rows, numbered through all slices, taken from `chains` runs of `chain` blocks by
// turns.  With a run about as long as a slice, work groups that follow each other read the same positions of different heads,
// which lie side by side.  A launch has chain * chains work groups, those past the last block have nothing to do.
template <typename Int>  // int or FmhaDivisor
FMHA_HOST_DEVICE int fmha_interleaved_block(int lin, int chain, const Int& chains) {
  const int step = lin / chains;
  return (lin - step * chains) * chain + step;
}
#endif  // FMHA_BLOCK_MAP_H_
