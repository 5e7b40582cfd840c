// How a split launch (prefill.hip) shares its workgroups between the prompts' tiles and the decode
// rows among them. Plain constexpr C++ that the host plan and the kernels compile, and a test on
// the CPU.
#pragma once

#include <stdint.h>

namespace nkv {

// Cost of one key step of a tile: its loads and the step's latency, and a share for each of
// its four waves that has rows to compute. With a smaller base (1 of 5) a range of a sequence's
// last, partial tile took up to twice the others' time: 1522 tokens in two chunks on 9000 (Hq 16,
// Hk 8) 207 us, with 5 of 9 155; three chunks and 10 decode rows 70.5, 65.1.
constexpr int kStepBase = 5;
constexpr int kFullStep = kStepBase + 4;

// Cost of a 16-key chunk of a decode row, in twentieths of a full tile's step: fewer workgroups
// than the rows' share of the time alone would give them (5 and 3), since the memory serves them
// at its full rate from half the chip's waves while the others compute. 48 rows with two
// 512-token chunks, at 1, 2, 3, 4, 6: 116, 117, 126, 129, 160 us; 80 rows of 4k - 8k with one:
// 333, 319, 316, 361; 60 fp8 rows with two: 88, 111, 119, 125.
constexpr int row_cost(bool f8) { return f8 ? 1 : 2; }

// The fewest workgroups of a KV head that the decode rows can have: each brings four waves, and
// every group of `hp` KV heads and every one of its `ncg` column groups of query heads needs a
// wave of its own (decode_stream.h).
constexpr int row_ranges_least(int ncg, int hp) { return (ncg + 4 * hp - 1) / (4 * hp); }

// Workgroups of each KV head for the decode rows and for the tiles.
struct SplitShare {
  int rows, tiles;
};
// n_ranges (more than row_ranges_least) workgroups of a KV head shared out by cost over `chunks`
// chunks of decode rows and tiles of `tile_cost`: each kind of work that there is has at least
// the fewest that do it, however little of it there is, since the rows are no tiles and only
// their own workgroups compute them.
constexpr SplitShare split_share(int n_ranges, int chunks, int tile_cost, bool f8, int ncg,
                                 int hp) {
  if (chunks <= 0) return SplitShare{0, n_ranges};
  if (tile_cost <= 0) return SplitShare{n_ranges, 0};
  const float cost = (float)chunks * ((float)(row_cost(f8) * kFullStep) / 20.f);
  const int r = (int)((float)n_ranges * cost / (cost + (float)tile_cost) + 0.5f);
  const int least = row_ranges_least(ncg, hp);
  const int rows = r < least ? least : r < n_ranges - 1 ? r : n_ranges - 1;
  return SplitShare{rows, n_ranges - rows};
}

// Whether a split launch's positions fit 32 bits with n_seqs sequences of up to `keys` keys (whose
// lengths are 32 bits) and `tiles` tiles of theirs: the tiles' key steps by cost, of which a range's
// end can lie as far past the last as a range is long, and the decode rows' chunks.
constexpr bool split_fits(int64_t n_seqs, int64_t tiles, int64_t keys) {
  constexpr int64_t most = 1000000000;
  if (n_seqs > most || tiles > most) return false;  // the products below stay within 64 bits
  if (keys > INT32_MAX) keys = INT32_MAX;
  const int64_t steps = keys > 64 ? (keys + 63) / 64 : 1;
  return tiles * steps * kFullStep <= most && n_seqs * ((keys + 15) / 16) <= most;
}

}  // namespace nkv
