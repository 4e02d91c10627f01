// How the launches of the last-query scores are cut (sp_scores.hip): host arithmetic on sizes, no device code.
#pragma once
#include <stdint.h>

#define LQ_WG_HEADS 2      // heads of one kv group a workgroup has
#define LQ_FOLD_CHUNKS 32  // chunks up to which the probabilities kernel folds them in its prologue instead: 16 loads per lane
#define LQ_MAX_TILES 32    // key tiles of 128 per workgroup of the statistics kernel, at most

static inline int64_t lq_ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
// rows of the grid: workgroups per key chunk.  A group with an odd head count leaves its last workgroup half empty.
static inline int lq_wg_rows(int hq, int hkv) { return hkv * (int)lq_ceil_div(hq / hkv, LQ_WG_HEADS); }

// Key tiles per workgroup of the statistics kernel: of all counts the one whose launch is the shortest, by the times it was measured
// to take (0.01 us; 128 channels, 3001 to 131072 tokens, counts 1 to 32, each within 10 %): a tile 2.9 us in a workgroup that has its CU
// to itself and 2.35 per tile of a CU with two, 6 and 9.5 us besides, and the launch that folds what the probabilities kernel does not
// fold itself; a CU without a workgroup counts 0.03 us, by what layers take (6177 tokens of 64 channels: 208 workgroups of four tiles
// 122.2 us, 400 of two 121.6).  Against counts that were powers of two and made some 512 workgroups, us for both: 4500 tokens
// 17.8 / 15.5, 10007 of 28 heads 24.1 / 19.4, 16384 30.6 / 27.6, 20000 of 64 channels 34.9 / 24.0, 65001 90.7 / 85.0.
// By the grid's rows: cut for half the heads, groups of odd size and heads without a group got a second, nearly empty round.  Scores, us,
// so / as it is: 28 / 4 heads 20000 tokens 94.9 / 78.0, 49000 185 / 163, 131072 426 / 410; 40 / 8 10007 80.4 / 68.6; 14 / 2 of 64
// channels 65001 106 / 99.6; 32 / 32 16384 98.8 / 94.9.  (Against the powers of two 14 / 2 of 64 stays 2.9 % behind at 131072, 177 / 182.)
static inline int lq_tiles_per_wg(int64_t tiles, int64_t wg_rows) {
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int t = 1; t <= LQ_MAX_TILES; ++t) {
    const int64_t chunks = lq_ceil_div(tiles, t), wgs = chunks * wg_rows, per_cu = (wgs + 255) >> 8;
    const int64_t cost = (per_cu == 1 ? 290 * t + 600 + 3 * (256 - wgs) : 235 * t * per_cu + 950 + 130 * (((per_cu + 1) >> 1) - 1)) +
                         (chunks > LQ_FOLD_CHUNKS ? 450 : 0);
    if (cost < best_cost) best_cost = cost, best = t;
  }
  return best;
}
// Chunks of the launch for hq heads of whatever grouping has the most of them: the workspace's size does not know the kv heads.  Groups of
// an even size have hq / 2 rows, those of an odd size (hq + hq / size) / 2.
static inline int64_t lq_max_chunks(int64_t tiles, int hq) {
  int64_t most = hq % 2 == 0 ? lq_ceil_div(tiles, lq_tiles_per_wg(tiles, hq / 2)) : 0;
  for (int group = 1; group <= hq; group += 2)
    if (hq % group == 0) {
      const int64_t chunks = lq_ceil_div(tiles, lq_tiles_per_wg(tiles, lq_wg_rows(hq, hq / group)));
      if (chunks > most) most = chunks;
    }
  return most;
}

// Tiles per workgroup of the probabilities kernel: the launch runs in ceil(workgroups / 256) rounds, one workgroup per CU, and a round
// takes 4.3 us a tile and 6 besides.
static inline int lq_probs_tiles_per_wg(int64_t tiles, int64_t wg_rows) {
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int t = 1; t <= 64; ++t) {
    const int64_t cost = lq_ceil_div(lq_ceil_div(tiles, t) * wg_rows, 256) * (10 * t + 14);
    if (cost < best_cost) best_cost = cost, best = t;
  }
  return best;
}
