// Tables of a step's launches that follow from its entries' row counts.
// Row tiles of the paged attention launches (pegainfer_paged_attention_opt): a tile is a run of token rows of one entry times a run of the
// query heads of one key/value head.  Chunks of long entries, for recurrences with a chunk form.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace ptiles {

constexpr int kGroupRows = 16;      // (token, query head) rows of one workgroup of the general attention kernels
// Wide tiles (64 or 32 rows) walk their keys in one workgroup; launches of fewer than kUnsplitGroups workgroups of 16-row tiles deal theirs
// to several, up to 512 in all.  Where the 16-row form is not split either, wide tiles win at any length: 16 heads over 4 key/value heads of
// 128, 128 tokens (128 workgroups of 16 rows, 32 of 64) alone 13.9 / 9.9 us, behind 4096 cached tokens 239 / 81, behind 16 384 904 / 293;
// 32 decoding requests of 64 heads over 4 behind 2048 tokens 126 / 44.  Where it is, they win up to about 670 keys (64 tokens) to 800 (96
// tokens): 64 tokens alone 18.8 / 8.4 us, behind 1024 cached tokens 25 / 30, behind 4096 53 / 96, behind 16 384 141 / 360; 8 decoding
// requests of 64 heads over 4 behind 8192 tokens 57 / 143.  There a step takes them while no row walks more than kWideKeys keys and they give
// kWideGroups workgroups.
constexpr int kUnsplitGroups = 128, kWideGroups = 32, kWideKeys = 640;
// Most workgroups that share a row tile's keys.  One past the row's last key tile ends at once, so a short context pays for its own only: one
// request of 16 heads over 4 behind 4000 tokens 26 -> 10 us with 64 instead of 16 (four tiles of 64 keys each, a quarter of the chip).
constexpr int kMaxSplits = 64;

// Every row of the step is wanted, in order (any decode step that asks for all its logits): the launch that closes the last layer norms the rows for
// the output table, and no launch of its own picks and norms them.  In a decode step of 4 to 8 rows that launch was 3.5 to 4.8 us of a step of 230 to
// 340, all of it latency; any other choice of rows still takes it.
inline bool all_wanted(const int32_t* want, int W, int T) {
  if (W != T) return false;
  for (int i = 0; i < W; ++i)
    if (want[i] != i) return false;
  return true;
}

inline size_t count(const int32_t* lens, int n, int per, int rows) {
  const int tpt = std::max(1, rows / per), cuts = (per + rows - 1) / rows;
  size_t c = 0;
  for (int i = 0; i < n; ++i) c += (size_t)((lens[i] + tpt - 1) / tpt) * cuts;
  return c;
}
// Rows of a tile, at least half full when wide.  kv: key/value heads of the launch (<= 0: it takes no wide tiles); keys: the most a row
// walks (INT_MAX where the choice must follow from the step's shape alone, as in a step that is captured).
inline int wide_rows(const int32_t* lens, int n, int T, int per, int kv, int keys) {
  if (keys > kWideKeys && (long)count(lens, n, per, kGroupRows) * kv < kUnsplitGroups) return kGroupRows;
  for (int rows : {64, 32}) {
    const long tiles = (long)count(lens, n, per, rows);
    if (tiles * kv >= kWideGroups && (long)T * per * 2 >= tiles * rows) return rows;
  }
  return kGroupRows;
}
// The latent attention's tiles: runs of up to `most` (token, head) rows of one entry; two columns, first row and rows.  begin(i): keys before entry i's
// rows.  A launch of more workgroups than the chip holds at once (one per compute unit) ends with the last to start, so the tiles of rows with the
// most keys go first, in steps of 64: prompts of 901, 701, 501 and 301 tokens, 16 heads of 512 + 64, 108 -> 99 us, one of 1800 180 -> 139, one of
// 4096 616 -> 538.  (The other attentions' prompts, whose workgroups are shorter and share a compute unit, lose by it: 1 % of whole runs.)
constexpr size_t kOrderedTiles = 64;     // fewer start together
inline size_t flat_count(const int32_t* lens, int n, int heads, int most) {
  size_t c = 0;
  for (int i = 0; i < n; ++i) c += ((size_t)lens[i] * heads + most - 1) / most;
  return c;
}
template <typename Begin>
inline void flat_cut(const int32_t* lens, int n, int heads, int most, size_t tiles, int32_t* table, Begin&& begin) {
  const bool ordered = tiles >= kOrderedTiles;
  auto each = [&](auto&& put) {
    int r0 = 0;
    for (int i = 0; i < n; r0 += lens[i++])
      for (int r = 0; r < lens[i] * heads; r += most) {
        const int rows = std::min(most, lens[i] * heads - r);
        put(r0 * heads + r, rows, ordered ? (size_t)(begin(i) + (r + rows - 1) / heads) >> 6 : 0);
      }
  };
  std::vector<size_t> left(1, 0);        // tiles of each step of keys, then the place of the next one
  each([&](int, int, size_t step) {
    if (step >= left.size()) left.resize(step + 1, 0);
    ++left[step];
  });
  size_t before = 0;
  for (size_t s = left.size(); s-- > 0;) {
    const size_t count = left[s];
    left[s] = before;
    before += count;
  }
  each([&](int row0, int rows, size_t step) {
    const size_t at = left[step]++;
    table[at] = row0;
    table[tiles + at] = rows;
  });
}
// the table's four columns, `tiles` (= count()) values each: first token row, tokens, first query head, query heads
inline void cut(const int32_t* lens, int n, int per, int rows, size_t tiles, int32_t* table) {
  int32_t *row0 = table, *ntok = row0 + tiles, *qh0 = ntok + tiles, *nqh = qh0 + tiles;
  const int tpt = std::max(1, rows / per);
  size_t at = 0;
  int r0 = 0;
  for (int i = 0; i < n; r0 += lens[i++])
    for (int t0 = 0; t0 < lens[i]; t0 += tpt)
      for (int q0 = 0; q0 < per; q0 += rows, ++at) {
        row0[at] = r0 + t0; ntok[at] = std::min(tpt, lens[i] - t0); qh0[at] = q0; nqh[at] = std::min(rows, per - q0);
      }
}

// Rows of a tile of the experts' table of a step of T rows.  Up to kFewRows rows the table is cut at T: the GEMMs of few rows take no
// more than that from a tile, and an expert can have more pairs than there are rows (a row that no expert is eligible for puts all its
// choices on one).  wide: the GEMMs walk tiles of 128 rows.
constexpr int kFewRows = 16;
inline int expert_tile_rows(int T, bool wide) { return T <= kFewRows ? T : wide ? 128 : 64; }
// most tiles of a step of T rows with `top` choices each: every tile holds a pair
inline int expert_tiles(int T, int top, int experts, int per_tile) {
  const int P = T * top;
  return std::min(P, (P + per_tile - 1) / per_tile + experts);
}

// Slices in which an expert that every row takes joins the routed ones' launches of few rows (0: it has launches of its own)
inline int shared_slices(int T, bool wide, int shared_ff, int ff) {
  return wide && T <= kFewRows && shared_ff > 0 && shared_ff % ff == 0 ? shared_ff / ff : 0;
}

// the chunks of the entries of more than scan_max rows (pegainfer_decay_attention's tables)
struct Chunks {
  std::vector<int32_t> row0, rows, first{0}, slot;     // per chunk; per long entry: its first chunk (one more at the end), its state slot
};
inline Chunks chunks(const int32_t* ids, const int32_t* lens, int n, int width, int scan_max) {
  Chunks c;
  for (int i = 0, r0 = 0; i < n; r0 += lens[i++]) {
    if (lens[i] <= scan_max) continue;
    for (int k = 0; k < lens[i]; k += width) {
      c.row0.push_back(r0 + k);
      c.rows.push_back(std::min(width, lens[i] - k));
    }
    c.first.push_back((int32_t)c.row0.size());
    c.slot.push_back(ids[i]);
  }
  return c;
}

}  // namespace ptiles
