// Rules by which launches are chosen and share out their work: the variable-length attention's
// (prefill.hip), a plain launch's tile size, and a split one's workgroups between the prompts'
// tiles and the decode rows among them; and the waves that merge a decode row (paged_decode.hip).
// Plain constexpr C++ that the host and the kernels compile, and a test on the CPU.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace nkv {

// What the host knows of a batch's composition: as few prompts as could bring its rows of q
// (total_q; every sequence's max_seqlen_q where it is not known), the others being decode rows.
struct BatchMix {
  int64_t prompts, rows, prompt_rows;  // prompts, decode rows, the prompts' rows of q
};
constexpr BatchMix batch_mix(int64_t n_seqs, int64_t total_q, int64_t max_seqlen_q) {
  if (total_q < 0) total_q = n_seqs * max_seqlen_q;
  const int64_t more = std::max<int64_t>(0, total_q - n_seqs);  // beyond one token each
  BatchMix m{};
  m.prompts = max_seqlen_q > 1
                  ? std::min(n_seqs, (more + max_seqlen_q - 2) / (max_seqlen_q - 1))
                  : 0;
  m.rows = n_seqs - m.prompts;
  m.prompt_rows = total_q - m.rows;
  return m;
}

// Tiles of qt queries a sequence in a plain launch's grid, enough for the longest: with more than one
// sequence an odd number. Most sequences of a mixed step have one tile (a decode row), every
// plain_tiles-th workgroup of a KV head, and workgroups go to XCDs and CUs in turn: a stride with
// powers of two in it leaves the work to a few of them. 250 rows of up to 500 keys and a prompt
// (Hq 32, Hk 8, 64 rows a tile, even / odd, us): of 120 tokens (8, 9 tiles) 199 / 78, of 500 (32,
// 33) 215 / 100; Hq 8, Hk 2: 145 / 31.
constexpr int64_t plain_tiles(int64_t n_seqs, int64_t max_seqlen_q, int64_t qt) {
  const int64_t tiles = (max_seqlen_q + qt - 1) / qt;
  return n_seqs > 1 ? tiles | 1 : tiles;
}

// Row groups per wave of a plain launch, up to `most` (every number gives the same bits). More rows
// a tile need fewer reads of K and V from LDS per MFMA, fewer leave more workgroups to overlap, and
// a workgroup's key step takes 1.15 us with one, 1.26 with two, 1.75 with three while the chip is
// not full. Measured (Hq 32, Hk 8; 1 / 2 / 3 groups, us; workgroups as with three):
//   a prompt of 333 (56 workgroups)     10.1 /  13.2 /  18.9
//   of 1500 (256)                       34.1 /  38.1 /  50.6
//   of 3000 (504)                      100.0 /  81.8 /  99.4
//   four chunks of 2048 on 6000 (1376)  1059 /   816 /   847
//   16 prompts up to 1500 (4224)         206 /   159 /   170
//   16 prompts up to 4096 (11136)       1206 /   933 /   925
//   250 decode rows, a prompt of 60      35.3 /  41.4 /  52.9 (a row's tile is a row)
// Large GQA groups g leave a part of a tile's rows unused, more of a small tile's (a group of 48
// fills 192 rows, 96 of 128): the lines lie at the tiles that there are of each size, and on a
// full chip two groups need 7/8 of the use that `most` makes of its rows (1 / 2 / 3, us):
//   Hq 33, Hk 1 (64, 99, 165 rows used): 600 15.1 / 17.7 / 25.0, 1300 44.9 / 33.2 / 44.3,
//     16 prompts up to 1500 168 / 97 / 102
//   Hq 48, Hk 1 (48, 96, 192): 1300 45.4 / 37.1 / 46.4, 2000 88.0 / 73.9 / 68.2, 6 of 1000 152 /
//     118 / 97
//   Hq 96, Hk 1 (-, 96, 192): 600 - / 23.8 / 28.0, 1300 - / 64.1 / 52.9, 6 of 1000 - / 235 / 180
constexpr int plain_groups(int64_t n_seqs, int64_t total_q, int64_t max_seqlen_q,
                           int32_t n_kv_heads, int g, int most, int cus) {
  const BatchMix m = batch_mix(n_seqs, total_q, max_seqlen_q);
  const auto queries = [&](int groups) -> int64_t { return 64 * groups / g; };  // of a tile
  const auto tiles = [&](int groups) -> int64_t {
    const int64_t qt = queries(groups);
    return std::min(m.prompts * ((max_seqlen_q + qt - 1) / qt), m.prompt_rows / qt + m.prompts);
  };
  // workgroups, tiles counted by their size
  const auto size = [&](int groups) -> int64_t {
    return (tiles(groups) * groups / most + m.rows) * n_kv_heads;
  };
  int want = most;
  if (g <= 64 && (size(1) <= cus || m.rows >= tiles(most))) {
    want = 1;
  } else if (most > 2) {
    const bool used = 8 * most * queries(2) >= 7 * 2 * queries(most);
    if (size(2) <= (used ? 16 : 2) * cus) want = 2;
  }
  // Every sequence's tiles are launched as for the longest, and each empty workgroup takes its turn:
  // the smaller sizes only while a launch stays small. 120 rows and 4 prompts of 500 (Hq 64, Hk 8;
  // 64480, 32736, 20832 workgroups): 89 / 69 / 70 us.
  const auto launched = [&](int groups) -> int64_t {
    return n_seqs * plain_tiles(n_seqs, max_seqlen_q, queries(groups)) * n_kv_heads;
  };
  if (want == 1 && launched(1) > 24576) want = std::min(most, 2);
  if (want == 2 && launched(2) > 49152) want = most;
  return want;
}

// Cost of one key step of a tile: its loads and the step's latency, and a share for each of
// its four waves that has rows to compute. With a smaller base (1 of 5) a range of a sequence's
// last, partial tile took up to twice the others' time: 1522 tokens in two chunks on 9000 (Hq 16,
// Hk 8) 207 us, with 5 of 9 155; three chunks and 10 decode rows 70.5, 65.1.
constexpr int kStepBase = 5;
constexpr int kFullStep = kStepBase + 4;

// Cost of a 16-key chunk of a decode row for one KV head, a full tile's step being kFullStep: fewer
// workgroups than the rows' share of the time alone would give them (5 / 20 and 3 / 20 of a step in
// bf16 and fp8 at head_dim 128), since the memory serves them at its full rate from half the
// chip's waves while the others compute. 48 rows with two 512-token chunks, at 1, 2, 3, 4, 6
// twentieths: 116, 117, 126, 129, 160 us; 80 rows of 4k - 8k with one: 333, 319, 316, 361; 60 fp8
// rows with two: 88, 111, 119, 125. At head_dim 256 a chunk is twice the bytes beside a step of a
// third of the rows, and each of `ncg` column groups streams it. Times over the best share's,
// geometric mean (worst), of random steps: 2 (bf16) and 1 (fp8) twentieths everywhere / as here
//   head_dim 256: 38 steps 1.10 (1.5) / 1.02 (1.1); fp8, 19 steps 1.30 (2.0) / 1.05 (1.3)
//   head_dim 128, four groups: 11 steps 1.18 (1.7) / 1.04 (1.1); fp8, 4 steps 1.36 / 1.17
//   head_dim 256, four groups: 6 steps 1.96 (2.7) / 1.03 (1.1)
constexpr float row_cost(int head_dim, bool f8, int ncg) {
  const int twentieths = head_dim == 256 ? (f8 ? 3 : 4) : (f8 ? 1 : 2);
  return (float)(twentieths * ncg * kFullStep) / 20.f;
}

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
constexpr SplitShare split_share(int n_ranges, int chunks, float chunk_cost, int tile_cost,
                                 int ncg, int hp) {
  if (chunks <= 0) return SplitShare{0, n_ranges};
  if (tile_cost <= 0) return SplitShare{n_ranges, 0};
  const float cost = (float)chunks * chunk_cost;
  const int r = (int)((float)n_ranges * cost / (cost + (float)tile_cost) + 0.5f);
  const int least = row_ranges_least(ncg, hp);
  const int rows = r < least ? least : r < n_ranges - 1 ? r : n_ranges - 1;
  return SplitShare{rows, n_ranges - rows};
}

// Whether a split launch's positions fit 32 bits with n_seqs sequences of up to `keys` keys (whose
// lengths are 32 bits) and `tiles` tiles of theirs: the tiles' key steps by cost, of which a
// range's end can lie as far past the last as a range is long, and the decode rows' chunks.
constexpr bool split_fits(int64_t n_seqs, int64_t tiles, int64_t keys) {
  constexpr int64_t most = 1000000000;
  if (n_seqs > most || tiles > most) return false;  // the products below stay within 64 bits
  if (keys > INT32_MAX) keys = INT32_MAX;
  const int64_t steps = keys > 64 ? (keys + 63) / 64 : 1;
  return tiles * steps * kFullStep <= most && n_seqs * ((keys + 15) / 16) <= most;
}

// Whether four waves merge the partials of a decode row instead of one: where a row may have more
// than 24, its sequence's share of the `waves` waves of each KV head and column group, or as many
// as a full table row makes (ranges of min_chunks of its max_chunks). One wave has 16 partials in
// flight at once and eight more in another round trip; four pay for their own merge (split
// and combine in a graph, one / four, us):
//   1 sequence of 16000 (Hq 32, Hk 8; up to 127)           23.6 /  16.5
//   3 of 1000 - 4000 (Hq 8, Hk 2; 87)                      16.2 /  11.4
//   12 of 4000 - 16000 (Hq 16, Hk 8; 23)                   88.6 /  84.5
//   100 of 250 - 1000 (Hq 16, Hk 1; 22)                    20.8 /  22.6
//   100 of 1000 - 4000 (Hq 80, Hk 1; 6)                   125.1 / 138.9
// Over 484 such shapes the line is nowhere slower than one wave alone, and 0.1% off the faster
// choice on average, 4.9% at most; from 16 partials on and with the column groups left out, 87
// of them were over 2% slower than one wave, up to 31%.
constexpr bool combine_wide(int64_t batch, int64_t n_kv_heads, int64_t ncg, int64_t max_chunks,
                            int64_t min_chunks, int64_t waves) {
  const int64_t share = waves / (n_kv_heads * ncg) / batch + 2;
  return std::min(share, (max_chunks + min_chunks - 1) / min_chunks + 1) > 24;
}

}  // namespace nkv
