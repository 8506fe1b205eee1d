// The prefill part's flat space of positions (see prefill_units in paged_attention.hip): plain
// integer functions of a sequence's lengths, shared by the kernels and compiled for the host by
// the test that compares them with a walk over every tile.
//
// A prefill-class sequence has R = q_len G query rows per kv head in ceil(R / PR) tiles of PR
// rows. Tile t occupies kTileCost + pre_tile_chunks positions: its fixed cost (query load, pipeline
// fill, output write), then the 32-key chunks its last row can see.
#pragma once
#include <stdint.h>

namespace kvh {

#ifndef KVH_PLAN_FN
#define KVH_PLAN_FN __device__ __forceinline__
#endif

constexpr int kPlanChunk = 32;  // keys of a chunk
// Fixed cost of a tile in chunk steps: each tile occupies kTileCost + chunks positions of the
// flat space, the first kTileCost virtual.
constexpr int kTileCost = 4;

// What the plan reads of a sequence: query rows R, the context before the step, the query
// length and the keys present (seq_len clamped to the block table's capacity).
struct PreSeq {
  int32_t R, q_len, kv_total;
  int64_t ctx;
};

// Chunks of tile t: those its last row can see, at least one so that every tile is visited
// and written.
KVH_PLAN_FN int pre_tile_chunks(const PreSeq& s, int G, int PR, int t) {
  const int end = PR * t + PR - 1, last = end < s.R - 1 ? end : s.R - 1;
  int64_t lim = s.ctx + last / G + 1;
  lim = lim < 0 ? 0 : (lim > s.kv_total ? s.kv_total : lim);
  const int c = (int)((lim + kPlanChunk - 1) / kPlanChunk);
  return c > 1 ? c : 1;
}

// floor(log2) of a power of two.
KVH_PLAN_FN int pre_log2(int x) { return __builtin_ctz((unsigned)x); }

// Positions of tiles 0 .. t - 1 of one kv head, t <= ceil(R / PR). With PR a multiple of G and
// no clamped length, a full tile i sees ctx + s (i + 1) keys (s = PR / G), so the sum of
// ceil((ctx + s i) / 32) over i = 1 .. n splits into whole chunks per tile and a remainder that
// repeats every 32 / gcd(s, 32) tiles (2 at PR = 192, G = 4): a few terms whatever the length
// of the prompt, and no division (step = PR / G, 0 when G does not divide PR). Any other case is
// added tile by tile.
KVH_PLAN_FN int64_t pre_prefix(const PreSeq& s, int G, int PR, int step, int t) {
  if (t <= 0) return 0;
  int64_t n = (int64_t)kTileCost * t;
  if (step > 0 && s.ctx >= 0 && s.ctx + s.q_len == s.kv_total) {
    const int tiles = s.R / PR, full = t < tiles ? t : tiles;
    const int a = step / kPlanChunk, b = step % kPlanChunk;
    const int64_t e = s.ctx + kPlanChunk - 1;
    const int e0 = (int)(e % kPlanChunk);
    n += full * (e / kPlanChunk) + (int64_t)a * full * (full + 1) / 2;
    const int lp = pre_log2(kPlanChunk) - pre_log2(b ? b & -b : kPlanChunk);  // log2 of the period
    const int per = (b << lp) / kPlanChunk;
    for (int r = 1; r <= 1 << lp && r <= full; ++r) {  // tiles r, r + period, ... (1-based)
      const int64_t m = ((full - r) >> lp) + 1;
      n += m * ((e0 + b * r) / kPlanChunk) + per * (m * (m - 1) / 2);
    }
    if (t > full) n += (s.kv_total + kPlanChunk - 1) / kPlanChunk;  // the last, partly filled tile
    return n;
  }
  for (int i = 0; i < t; ++i) n += pre_tile_chunks(s, G, PR, i);
  return n;
}

}  // namespace kvh
