// attn_plan.cpp — how launch_attention splits the work of the partitioned
// (long-sequence and batch) attention kernels, and the scratch that split
// needs: host arithmetic only, shared by the launcher, the model's workspace
// sizing and the argument checks.
#include "internal.hpp"

namespace glypr {

namespace {

// The most key tiles a block of `queries` query rows meets.
int64_t key_tiles(int64_t Tseg, int64_t window, int64_t queries) {
  int64_t nkb = (Tseg + ATTN_AK - 1) / ATTN_AK;
  if (window > 0 && Tseg > window) {
    const int64_t band = (2 * window + queries + ATTN_AK - 1) / ATTN_AK + 1;
    if (band < nkb) nkb = band;
  }
  return nkb;
}

// Sets the cheapest of 1 .. most partitions over nkb key tiles for `blocks`
// workgroups per partition and returns its cost in microseconds: every round
// of 256 workgroups (one per CU: the K/V ring or the accumulators leave room
// for one; two of two waves at head_dim 256 fit and count as one) takes `start`
// (launch, Q, first tile, epilogue) plus `tile` per key tile (`tile_full` past 60 %
// of the CUs: shared L2 reads, clocks), and a split pays for the combine launch and
// the f32 partials, written and read by the combine at ~8.7 TB/s (past 34 MB, which
// the caches do not hold, at 5.7).  A grid that fills a round by itself is never
// split.
double plan_parts(AttnPlan& p, int64_t blocks, int64_t nkb, double start, double tile,
                  double tile_full, int64_t part_bytes) {
  const double mb = part_bytes * 1e-6;
  double best = 0;
  int64_t most = nkb < ATTN_MAX_PARTS ? nkb : ATTN_MAX_PARTS;
  if (blocks >= ATTN_BLOCKS) most = 1;
  for (int64_t want = 1; want <= most; want++) {
    const double out = want * mb;
    const double split = want > 1 ? 1.2 + out * 0.23 + (out > 34 ? (out - 34) * 0.12 : 0.0) : 0.0;
    if (want > 1 && start + split >= best) break;   // so do all that follow
    const int64_t per = (nkb + want - 1) / want;
    if ((nkb + per - 1) / per != want) continue;
    const int64_t rounds = (blocks * want + ATTN_BLOCKS - 1) / ATTN_BLOCKS;
    const bool full = blocks * want * 5 > ATTN_BLOCKS * 3;
    const double c = rounds * (start + per * (full ? tile_full : tile)) + split;
    if (want == 1 || c < best) {
      best = c;
      p.per = (int)per;
      p.kparts = (int)want;
    }
  }
  return best;
}

}  // namespace

// The short kernel's grid is nkv Tp / 16 query rows wide and each of its
// workgroups walks all T keys alone.  On one kv head that wins up to 1024 rows; more
// heads fill the CUs several times over, and the partitioned kernels win from
// 1280 rows of all heads (2 x 2 heads: T = 640, 26.5 against 27.1 us; 850, 40.7
// against 30.3), unless the walks are short: nkv Tp Tp up to 600,000 (4 x 1 heads:
// T = 321, 18.5 against 21.4; 512, 28.0 against 24.8; 8 x 1: T = 200, 19.3 against
// 20.8; 321, 32.0 against 26.0).
bool attn_short(int64_t Tp, int64_t hd, int64_t nq, int64_t nkv, bool segments) {
  return hd == 256 && !segments && Tp <= 1024 && nq / nkv <= 3 &&
         (nkv * Tp <= 1280 || nkv * Tp * Tp <= 600000);
}

// The choices with their starts and tile times (us), fitted to every choice and
// partition count measured at 587 shapes (64 to 8192 keys, 1 to 8 kv heads of 1 to 4
// q heads, single sequences and batches); the chosen ones are 0.4 % slower than the
// best on average:
//   16-query blocks: few keys;
//   64-query blocks (head_dim 256): on few q heads, and where they fill just one
//     round and the 32 x 32 tiles leave SIMDs idle (32 sequences x 512 rows of 3
//     heads: 39.9 against 55.2 us; T = 8192 of 3 heads: 248 against 268 us; 64
//     sequences x 128 rows of 2 x 2 heads: 16.3 against 18.0);
//   32 x 32 tiles: everything longer (T = 1777, window 512: 49.9 -> 37.2 us with the
//     prologue; T = 3500 of 3 heads: 82 -> 69; T = 4000 of 4 heads, head_dim 512: 375
//     -> 185; T = 8192: 1472 -> 594).
AttnPlan attn_plan(int64_t Tseg, int64_t rows, int64_t hd, int64_t nq, int64_t nkv,
                   int64_t window, bool segments) {
  const int64_t G = nq / nkv, part_bytes = rows * nq * hd * 4;
  AttnPlan best{};
  double best_cost = 0;
  auto offer = [&](int waves, int qs, int64_t queries, int64_t blocks, double start,
                   double tile, double tile_full, int fit = 1) {
    AttnPlan p{waves, qs, 0, 0};
    const double c = plan_parts(p, (nkv * blocks + fit - 1) / fit,
                                key_tiles(Tseg, window, queries), start, tile, tile_full,
                                part_bytes);
    if (best.kparts == 0 || c < best_cost) {
      best = p;
      best_cost = c;
    }
  };
  const bool wide = hd == 512;
  if (wide) {
    offer(0, 1, 16, rows / 16, 2.1, 2.25, 2.25);
  } else {
    offer(0, 1, 16, rows / 16, 6.3, 0.84, 0.89);
    // (16 waves share the tiles at 4 heads: far slower once the CUs are full)
    offer(0, 4, 64, rows / 64, 6.6, 0.85 * G, G < 4 ? 1.0 : 5.0);
  }
  // Four column groups (32 queries of one head) per workgroup fill its CU's
  // SIMDs.  With several sequences a workgroup stays within one, so within 64
  // rows: two groups of one head, three of three heads.
  const int waves = !segments || G % 2 == 0 ? 4 : G == 1 ? 2 : 3;
  const int64_t queries = waves % G == 0 ? 32 * (waves / G) : 64;
  offer(waves, 0, queries, ((rows >> 5) * G + waves - 1) / waves, wide ? 4.8 : 8.8,
        wide ? 2.0 : 0.77, wide ? 1.72 : 0.68, waves == 2 && !wide ? 2 : 1);
  return best;
}

bool attention_rows_ok(int64_t rows, int64_t hd) {
  return 2 * hd * attn_padded_len(rows) < (int64_t(1) << 31);
}

bool attention_supported(int64_t T, int64_t nq, int64_t nkv, int64_t hd, int64_t window) {
  if ((hd != 256 && hd != 512) || nq <= 0 || nkv <= 0 || nq % nkv != 0 || nq / nkv > 4)
    return false;
  if (T <= 0) return true;
  if (!attention_rows_ok(T, hd)) return false;
  // A block's keys: at most 64 partitions (the combine holds one per lane) of 64
  // key tiles, 131,072 keys
  return key_tiles(T, window, hd == 512 ? 16 : 64) <= ATTN_MAX_PARTS * 64;
}

size_t attention_scratch_floats(int64_t T, int64_t nq, int64_t nkv, int64_t hd, int64_t window,
                                int64_t rows) {
  const int64_t tp = rows > 0 ? rows : attn_padded_len(T);
  int kp = attn_plan(T, tp, hd, nq, nkv, window, false).kparts;
  if (nq / nkv % 2 != 0) {   // segments change the plan of 1 and 3 heads only
    const int k = attn_plan(T, tp, hd, nq, nkv, window, true).kparts;
    kp = k > kp ? k : kp;
  }
  return (size_t)(kp * tp * nq * (hd + 2));
}

size_t attention_scratch_bound(int64_t max_t, int64_t cap_rows, int64_t nq, int64_t nkv,
                               int64_t hd, int64_t window) {
  // For one tk, the plan depends on rows only through the block counts and the
  // partials' bytes.  Every row count is visited until the coarsest blocks (128
  // queries: four groups of one head) fill a round by themselves: from there no choice
  // splits, and kparts * rows = rows peaks at the capacity.
  size_t best = 0;
  for (int64_t tk = 32;; tk += 32) {
    if (tk > max_t) tk = max_t;
    for (int64_t rows = attn_padded_len(tk); rows <= cap_rows; rows += 64) {
      size_t sc = attention_scratch_floats(tk, nq, nkv, hd, window, rows);
      best = sc > best ? sc : best;
      if (rows / 128 * nkv >= ATTN_BLOCKS && rows < cap_rows) {
        sc = attention_scratch_floats(tk, nq, nkv, hd, window, cap_rows);
        best = sc > best ? sc : best;
        break;
      }
    }
    // (past the widest band every tk plans alike, over fewer row counts)
    if (tk == max_t || (window > 0 && key_tiles(tk, window, 128) * ATTN_AK < tk)) break;
  }
  return best;
}

}  // namespace glypr
