// Which kernel a product of several rows takes, from its sizes alone (host
// code: no HIP, so that a test can compile it by itself).
//
// Two forms compute the same bits. A wave a tile (gemm_ranges) chains a
// tile's 32 K-ranges one after another, two or four at a time: its time is
// that chain while its waves find SIMDs of their own, then grows with the
// rounds its workgroups take over the 256 CUs. A pass a wave
// (pass_tiles_kernel) spreads the chain over eight waves: its time grows
// with its tiles from the first, and each costs more than a wave's share of
// a full chip. So the second wins where the first leaves the chip idle or
// its last round nearly empty, and nowhere else: Q8_0, 8,176 rows, K = 4,096
// take 130 and 85 us at 32 tokens, 343 and 622 at 512; Q4_0, 1,152 rows,
// K = 6,912 (down), 122 and 107 at 512, 93 and 94 at 448, 50 and 14 at 32.
//
// The estimates below are least-squares fits to 2,592 measured products
// (three formats, K 1,024 to 16,384, 256 to 8,176 rows, 17 to 512 tokens),
// within 3% of a wave a tile's time on average and 5 to 12% of a pass a
// wave's. Choosing by them is within 3% of a wave a tile alone in all but 17
// (10% at worst), and takes up to a quarter of its time.

#pragma once

#include <algorithm>
#include <cstdint>

namespace frz {
namespace rules {

constexpr int kRanges = 32;
constexpr int kCus = 256, kSimds = 1024;

constexpr int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Groups of K in range r.
constexpr int range_groups(int r, int groups) {
  return (r + 1) * groups / kRanges - r * groups / kRanges;
}

// The steps of a wave that chains the ranges in order, `blocks` at a time,
// each turn as long as its longest range.
inline int chain_steps(int groups, int blocks) {
  int steps = 0;
  for (int r = 0; r < kRanges; r += blocks) {
    int longest = 0;
    for (int b = 0; b < blocks; ++b) longest = std::max(longest, range_groups(r + b, groups));
    steps += longest;
  }
  return steps;
}

// The steps of a tile's passes of four ranges, longest ranges first.
constexpr int pass_steps(int groups) {
  return kRanges / 4 * (groups / kRanges) + ceil_div(groups % kRanges, 4);
}

// Straight-line forms of at most two steps a pass cost a tile less than the
// loop over longer ones.
constexpr int kShortGroups = 2 * kRanges;

// A wave a tile takes 32 x 32 tiles (two ranges in flight) when they cover
// most of the SIMDs, else 16 x 16 (four ranges), four times as many; 16
// tokens or fewer would waste half a 32 x 32 tile's columns.
inline bool wide_chain(int rows, int tokens) {
  return (int64_t)rows * tokens >= (int64_t)768 * 1024 && tokens > 16;
}

// Microseconds of a plain product, a pass a wave.
inline double pass_us(bool q4_0, int rows, int groups, int tokens) {
  const double tiles = (double)ceil_div(rows, 16) * ceil_div(tokens, 16) / kSimds;
  const int steps = pass_steps(groups);
  if (groups <= kShortGroups) return (q4_0 ? 3.7 + 0.71 * steps : 5.1 + 0.74 * steps) * tiles;
  return (q4_0 ? 10.9 + 0.77 * steps : 11.0 + 0.86 * steps) * tiles;
}

// The same, a wave a tile, four waves along the tokens a workgroup.
inline double chain_us(int rows, int groups, int tokens) {
  const bool wide = wide_chain(rows, tokens);
  const int dim = wide ? 32 : 16, row_tiles = ceil_div(rows, dim);
  const double rounds = ceil_div(row_tiles * ceil_div(tokens, 4 * dim), kCus);
  const double waves = (double)row_tiles * ceil_div(tokens, dim) / kSimds;
  const int steps = chain_steps(groups, wide ? 2 : 4);
  return wide ? 14.5 + steps * (0.20 + 0.76 * rounds + 0.47 * waves)
              : 7.5 + steps * (0.26 + 0.45 * rounds + 0.21 * waves);
}

// Products of 2 to 512 tokens whose ranges each hold a group: a pass a wave
// up to 16 tokens (a chain of 32 ranges would be one wave of each workgroup);
// past them, matrices of under 8,192 rows (a vocabulary's thousands of tiles
// fill the chip a wave a tile) where it is sooner.
inline bool takes_pass(bool q4_0, int rows, int groups, int tokens) {
  if (groups < kRanges) return false;
  if (tokens <= 16) return true;
  return rows < 8192 && pass_us(q4_0, rows, groups, tokens) <= chain_us(rows, groups, tokens);
}

// ---- gated products ---------------------------------------------------------

// The wide tiles' neurons (their span: 128 tokens). Tiles of 32 read half the
// LDS a product of tiles of 16; but a CU takes whole tiles, and where its last
// would be at most half of one, tiles of 16 leave it half idle for half the
// time. Of 32 and of 16 took 199 and 193 us at 512 rows of 6,912 neurons (K =
// 1,152; 3.4 tiles a CU), 149 and 162 at 384 (2.5), 206 and 223 for 8,192
// neurons at 512 (4).
inline int wide_dim(int rows, int tokens) {
  const int tiles = ceil_div(rows, 32) * ceil_div(tokens, 128);
  return ceil_div(tiles, kCus / 2) < 2 * ceil_div(tiles, kCus) ? 16 : 32;
}

// Microseconds in the three forms: a pass a wave, the wide tiles, and a wave
// a tile of two ranges at a time; fits to 2,346 measured products (K 1,024 to
// 16,384, 64 to 16,384 neurons, 17 to 512 tokens), within 5 to 6% on average.
// Choosing by them is within 3% of a wave a tile alone in all but 35 of 2,944
// (12% at worst, K = 16,384).
inline double gated_pass_us(int rows, int groups, int tokens) {
  const double tiles = (double)ceil_div(rows, 16) * ceil_div(tokens, 16) / kSimds;
  const int steps = pass_steps(groups);
  return (groups <= kShortGroups ? 7.1 + 1.22 * steps : 5.6 + 1.95 * steps) * tiles;
}

inline double gated_wide_us(int rows, int groups, int tokens) {
  const int tiles = ceil_div(rows, 32) * ceil_div(tokens, 128);
  const double rounds =
      wide_dim(rows, tokens) == 16 ? 0.5 * ceil_div(tiles, kCus / 2) : ceil_div(tiles, kCus);
  const double waves = (double)ceil_div(rows, 32) * ceil_div(tokens, 32) / kSimds;
  return 10.0 + groups * (0.31 + 0.75 * rounds + 0.41 * waves);
}

inline double gated_chain_us(int rows, int groups, int tokens) {
  const int row_tiles = ceil_div(rows, 32);
  const double rounds = ceil_div(row_tiles * ceil_div(tokens, 128), kCus);
  const double waves = (double)row_tiles * ceil_div(tokens, 32) / kSimds;
  return 12.0 + chain_steps(groups, 2) * (0.57 + 1.41 * rounds + 0.89 * waves);
}

enum class Gated { kWide, kPass, kChain };

// A pass a wave up to 16 tokens and wherever it is sooner than the better of
// the others. Of those, the wide tiles gain by chaining one range at a time:
// none of a pair waits for a longer one (6,912 neurons, K = 1,152 at 512
// rows: 219 us a wave a tile, 193 wide). Where the ranges are of one length
// and long nothing is waited for, and a wave a tile, with no barrier, is
// 3 to 10% sooner (6,912 neurons, K = 4,096: 321 and 333 us at 256 rows).
inline Gated gated_form(int rows, int groups, int tokens) {
  if (groups < kRanges) return Gated::kWide;
  if (tokens <= 16) return Gated::kPass;
  const bool chain = groups % kRanges == 0 && groups >= 4 * kRanges;
  const double other =
      chain ? gated_chain_us(rows, groups, tokens) : gated_wide_us(rows, groups, tokens);
  if (gated_pass_us(rows, groups, tokens) <= other) return Gated::kPass;
  return chain ? Gated::kChain : Gated::kWide;
}

}  // namespace rules
}  // namespace frz
