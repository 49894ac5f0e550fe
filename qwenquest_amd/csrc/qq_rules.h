// The integer rules by which the launches divide their work: what the host sizes a grid
// and a workspace by, and what the kernels find their share by.  Plain constexpr
// functions, so that both sides, and a host compiler, run the same ones.
#pragma once

#include <stdint.h>

namespace qq {
namespace rules {

constexpr int64_t least(int64_t a, int64_t b) { return a < b ? a : b; }
constexpr int64_t most(int64_t a, int64_t b) { return a > b ? a : b; }
constexpr int64_t ceil_of(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ------------------------------------------------- unit attention (Quest step)
constexpr int kUnitParts = 8;  // blocks per (request, KV head), at most: merged in one pass

// Launch shape of the unit attention: W waves per block, `parts` blocks per (request,
// KV head); wave w of part p takes the units w * parts + p, + W * parts, ... one after
// the other.  The grid is sized to one round of resident blocks, since each block pays
// its own selection, row lookups and merge before and after its streaming (us per
// layer-step, top_k 2048 at 4 KV heads unless said):
//  * a unit per wave in 4-wave blocks that leave each CU at most one: those (batch 8:
//    16.4, 18.2 in 8-wave blocks; batch 9, where they would be more than the CUs: 19.9
//    against 18.7);
//  * up to one pair per CU: 8-wave blocks (one per CU), parts = CUs / pairs, unless two
//    4-wave blocks per CU, parts = 2 CUs / pairs, leave a wave fewer units in a row
//    (batch 34: 42.3 in 4-wave blocks, three parts, against 47.6; batch 40: 45.5 and
//    48.1, at top_k 4096 75.9 and 83.9; batch 48, where the rows are as long: 51.7
//    and 50.5);
//  * more pairs: 4-wave blocks, 3 parts up to 4/3 pairs per CU, then 2, past 8/5 1
//    (batch 72: 74.3 in 3, 77.1 in 2; batch 84: 81.4 and 83.0; batch 96: 94.7 and 89.6;
//    batch 104: 102.2 in 2, 96.3 in 1), but no part that leaves the longest wave as many
//    units (top_k 1024, 2 units a wave in 2 parts and in 3: batch 84 51.4 us in 3, 49.8 in 2).
// A second round of units in a part is dealt over all parts, not to the first ones
// (batch 20, 32 units over 24 waves: 32.0 -> 28.5; choosing the order by whether there
// is a second round costs batch 1 more, 0.04 us a layer, than the order does).
struct UnitShape {
  int W, parts;
};
constexpr UnitShape unit_shape(int64_t cus, int64_t bs, int kv_heads, int top_k) {
  const int64_t units = top_k / 64, pairs = bs * kv_heads;
  const int64_t cap8 = most(1, least(kUnitParts, ceil_of(units, 8)));
  const int64_t cap4 = most(1, least(kUnitParts, ceil_of(units, 4)));
  if (units <= 4 * cap4 && pairs * cap4 <= cus) return {4, (int)cap4};
  if (pairs <= cus) {
    const int64_t p8 = most(1, least(cap8, cus / pairs));
    const int64_t p4 = most(1, least(cap4, 2 * cus / pairs));
    if (ceil_of(units, 4 * p4) < ceil_of(units, 8 * p8)) return {4, (int)p4};
    return {8, (int)p8};
  }
  const int64_t parts = least(cap4, 3 * pairs <= 4 * cus ? 3 : 5 * pairs <= 8 * cus ? 2 : 1);
  return {4, (int)ceil_of(units, 4 * ceil_of(units, 4 * parts))};
}

// The units of wave `wave` of part `part`: this one, + W * parts, ...
constexpr int unit_first(int wave, int part, int parts) { return wave * parts + part; }

// ------------------------------------------------------------- dense decode
// A (request, KV head) pair's 64-row units are split into equal parts, one to a block;
// a CU holds one block.  Per KV head, `round` blocks are resident at once.
constexpr int kDenseKV = 4;        // KV heads of the dense decode kernel (KV*D = 512)
constexpr int kDenseBlocks = 256;  // blocks of a round, at most
constexpr int kDenseParts = 64;    // parts of a pair, at most: the merge's table of weights
constexpr int kDenseWhole = 8;     // units of a pair that is not split
constexpr int kDenseMinLen = 2;    // units of a part, at least

// Units of 64 rows; a request without rows has one, which writes its zeros.
constexpr int dense_units(int rows) { return (int)most((rows + 63) / 64, 1); }

// Parts of a pair for parts of `len` units.  A pair of up to a unit per wave stays
// whole, which saves its merge (one request of 500 rows: 12.9 us against 15.3 in two
// parts); longer ones may go down to two units a part (four of 1000 rows: 16.5 us, at
// four units 17.4, at eight 19.6; one of 8000: 18.0, 17.8 and 19.9).
constexpr int dense_parts(int units, int len) {
  return units <= kDenseWhole ? 1 : (int)least((units + len - 1) / len, kDenseParts);
}

// First unit of part `part` of `parts` of a pair: equal parts.
constexpr int dense_part_begin(int units, int part, int parts) { return (int)((int64_t)units * part / parts); }

constexpr int dense_round(int64_t cus) { return (int)most(least(cus, kDenseBlocks) / kDenseKV, 1); }

// Batches that one round of blocks always divides well enough: parts of `len` units fit
// a round from len = total / (round - bs) on, and a CU alone reads 8/5 of its share of
// the chip's rate (36 GB/s of 22.6), so that parts of up to 8/5 of the mean cost nothing:
// up to 3/8 of the round's parts.
constexpr bool dense_one_round(int64_t bs, int round) { return 8 * bs <= 3 * (int64_t)round; }

// Parts per KV head that the grid holds (it is sized without the lengths, which are on
// the device): one round, or for larger batches one part per request and two rounds'
// more, with which any batch divides into parts of half the mean; no more than the
// table's width can need.  An entry without work is a block that exits.
constexpr int64_t dense_fit(int64_t cus, int64_t bs, int64_t max_rows) {
  const int64_t units = most(ceil_of(max_rows, 64), 1), round = dense_round(cus);
  if (units <= kDenseWhole) return bs;
  if (dense_one_round(bs, (int)round)) return most(bs, least(round, bs * units));
  return bs + least(2 * round, bs * (ceil_of(units, kDenseMinLen) - 1));
}

// The part lengths that are tried, 64 from lo to hi, for `total` units per KV head of
// which one pair has `longest`; fit > bs.  (32-bit, as one block computes it before the
// attention can start; a total above kDenseMaxTotal stands for more, and dense_cost then
// finds the lengths that do not fit.)
constexpr int kDenseMaxTotal = 1 << 24;
struct DenseRange {
  int lo, hi;
};
constexpr int ceil32(int a, int b) { return (a + b - 1) / b; }
constexpr int least32(int a, int b) { return a < b ? a : b; }
constexpr int most32(int a, int b) { return a > b ? a : b; }
constexpr DenseRange dense_range(int total, int longest, int bs, int fit, int round) {
  if (dense_one_round(bs, round)) {
    const int lo = most32(ceil32(total, fit), kDenseMinLen);
    return {lo, most32(lo, least32(longest, ceil32(total, fit - bs)))};  // sum of ceil(u / hi) <= fit
  }
  const int lo = most32(ceil32(total, fit - bs), kDenseMinLen);  // sum of ceil(u / lo) <= fit
  int hi = least32(longest, 4 * ceil32(total, round));
  if (bs < round) hi = least32(hi, ceil32(total, round - bs));  // fits one round
  return {lo, most32(lo, hi)};
}
constexpr int dense_candidate(DenseRange r, int lane) { return r.lo + (r.hi - r.lo) * lane / 63; }

// What a division into `count` parts of up to `len` units costs, in the time that the
// chip at its full rate takes for one unit per block: the whole at that rate, or 5/8 of
// the longest run of parts on a CU, which reads that much faster alone, and six units
// (about 9 us) for the start and end of each block on it.  The first of the cheapest
// lengths is taken; where none fits, no pair is split.  (It takes halves for 70 x 10000
// rows, 311 us against 342 in whole pairs, and for 65 x 3000, 110 against 111.)
constexpr float kDenseNoFit = 1e30f;
constexpr float dense_run(int total, int count, int len, int round) {  // 5/8 of the longest run on a CU
  const float rounds = (float)ceil32(count, round), even = rounds * (float)total / (float)count;
  return 0.625f * (rounds > 1.0f && even > (float)len ? even : (float)len);
}
constexpr float dense_cost(int total, int count, int len, int fit, int round) {
  if (count > fit) return kDenseNoFit;
  const float run = dense_run(total, count, len, round), mean = (float)total / (float)round;
  return (run > mean ? run : mean) + 6.0f * (float)ceil32(count, round);
}

// No pair is split where that cannot cost more than any division: short pairs, or a run
// of whole ones that the chip's rate hides.  (The lengths are then not tried, which the
// attention waits for: 3.5 us at 128 requests, 9 at 300.)
constexpr bool dense_all_whole(int total, int longest, int bs, int round) {
  return longest <= kDenseWhole || dense_run(total, bs, longest, round) <= (float)total / (float)round;
}

// Where the parts take more than one round, those longer than half the part length come
// first, so that a round's end does not wait for a long one.
constexpr bool dense_first(int units, int parts, int len) { return 2 * ((units + parts - 1) / parts) > len; }

// ------------------------------------------------------------------ prefill
constexpr int kExtRows = 128;      // query rows per block
constexpr int kExtTile = 64;       // tokens per K/V tile
constexpr int kExtMinChunk = 4;    // K/V tiles that are worth a split
constexpr int kExtMaxSplits = 32;

// Query tiles of n tokens in bs requests, at most: every request's last tile may
// be partial.
constexpr int64_t extend_tiles(int64_t n, int64_t bs, int G) { return n * G / kExtRows + bs; }

// Tiles of one request.
constexpr int extend_request_tiles(int64_t n, int G) { return (int)((n * G + kExtRows - 1) / kExtRows); }

// K/V splits: as many as give every CU a block when the query tiles do not, one for
// every kExtMinChunk K/V tiles at most.  The merge costs a launch (6 us), so a grid that
// covers half the chip stays whole.  Us a call: 600 new tokens (152 blocks) 30.5, in two
// splits 34.6; 8 new tokens behind 8192 (4 blocks) in 32 splits 26.0, in 9 of 16
// tiles 44.9; 64 behind 8192 (16 blocks) in 12 splits 42.2, in 25 52.9.  A minimum of 4
// tiles against 8 and 16: 100 new behind 500, one KV head, 21 against 28 us.
constexpr int extend_splits(int64_t tiles, int KV, int64_t max_rows) {
  const int64_t by_grid = 256 / most(tiles * KV, 1);
  const int64_t by_rows = ceil_of(max_rows, kExtTile * kExtMinChunk);
  return (int)most(1, least(least(by_grid, by_rows), kExtMaxSplits));
}

// K/V tiles per split of a query tile that attends nt of them: equal parts, at most one
// for every kExtMinChunk.
constexpr int split_chunk(int nt, int splits) {
  const int64_t parts = most(least(splits, ceil_of(nt, kExtMinChunk)), 1);
  return (int)most(ceil_of(nt, parts), 1);
}

}  // namespace rules
}  // namespace qq
