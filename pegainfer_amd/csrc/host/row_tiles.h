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
// A step whose 64- (32-) row tiles give so many workgroups takes those; below, 16-row tiles whose keys are dealt to several workgroups have more
// of them.  16 heads over 4 key/value heads of 128, 16 / 32 / 64 rows: 1024 tokens 82 / 38 / 28 us, 128 tokens (32 workgroups of 64 rows)
// 14.5 / 10.4 / 10.2 us, behind 2048 cached tokens 128 / 55 / 45 us.
constexpr int kWideGroups = 32;

inline size_t count(const int32_t* lens, int n, int per, int rows) {
  const int tpt = std::max(1, rows / per), cuts = (per + rows - 1) / rows;
  size_t c = 0;
  for (int i = 0; i < n; ++i) c += (size_t)((lens[i] + tpt - 1) / tpt) * cuts;
  return c;
}
// rows of a tile for a step of prompts: the widest tiles that still fill the chip (kv: key/value heads of the launch; <= 0: the launch
// takes no wide tiles) and are at least half full
inline int wide_rows(const int32_t* lens, int n, int T, int per, int kv) {
  for (int rows : {64, 32}) {
    const long tiles = (long)count(lens, n, per, rows);
    if (tiles * kv >= kWideGroups && (long)T * per * 2 >= tiles * rows) return rows;
  }
  return kGroupRows;
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
