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

// The greatest common divisor of two positive numbers.
KVH_PLAN_FN int pre_gcd(int a, int b) {
  while (b) {
    const int r = a % b;
    a = b;
    b = r;
  }
  return a;
}

// Positions of tiles 0 .. t - 1 of one kv head, t <= ceil(R / PR). With no clamped length, full
// tile i (from 1) sees ctx + ceil(PR i / G) keys, ceil((ctx G + PR i) / (32 G)) chunks, and the sum over
// i = 1 .. n splits into whole chunks per tile and a remainder that repeats after a few tiles: a few
// terms whatever the length of the prompt.
//  * step = PR / G where G divides PR: the remainder is that of (ctx + step i) / 32 and repeats every
//    32 / gcd(step, 32) tiles (2 at PR = 192, G = 4), with no division.
//  * step = 0, G does not divide PR (groups of 5, 7 or 10; of 3 and 6 at PR = 128): every 32 G /
//    gcd(PR, 32 G) tiles, at most G. A walk from the first tile instead made the search for a unit's
//    start quadratic in the prompt: 32768 tokens, G = 7, E4M3 caches, 11466 us against 8313.
// A clamped length is added tile by tile.
KVH_PLAN_FN int64_t pre_prefix(const PreSeq& s, int G, int PR, int step, int t) {
  if (t <= 0) return 0;
  int64_t n = (int64_t)kTileCost * t;
  if (s.ctx < 0 || s.ctx + s.q_len != s.kv_total) {
    for (int i = 0; i < t; ++i) n += pre_tile_chunks(s, G, PR, i);
    return n;
  }
  const int tiles = s.R / PR, full = t < tiles ? t : tiles;
  if (step > 0) {
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
  } else {
    const int M = kPlanChunk * G, g = pre_gcd(PR, M), period = M / g, per = PR / g;
    const int a = PR / M, b = PR % M, whole = full / period, left = full % period;
    int q = 0, rem = (int)(s.ctx % kPlanChunk) * G + M - 1;  // below 2 M
    if (rem >= M) {
      rem -= M;
      q = 1;
    }
    n += full * (s.ctx / kPlanChunk);
    for (int r = 1; r <= period && r <= full; ++r) {  // tiles r, r + period, ...; q chunks of tile r
      q += a;
      rem += b;
      if (rem >= M) {
        rem -= M;
        ++q;
      }
      const int64_t m = whole + (r <= left);
      n += m * q + per * (m * (m - 1) / 2);
    }
  }
  if (t > full) n += (s.kv_total + kPlanChunk - 1) / kPlanChunk;  // the last, partly filled tile
  return n;
}

}  // namespace kvh
