// Which form of the skinny GEMM (skinny.h) a weight takes, and how k is split: plain functions of its
// shape and the rows of x, also compiled for the host by the test that holds them to what was measured.
#pragma once
#include <stdint.h>

namespace kvh {

constexpr int kSkinnyWaves = 8;       // waves of a workgroup: `ks` for each of its tiles
enum SkinnyForm { kSkinnyFull, kSkinnyHalf, kSkinnyShared };

// The form of a weight of `rows` rows: a function of its shape and of m alone, so that a projection and
// its fused forms sum in one order. Times in us, (rows, k) at m rows of x, cold weights, bf16:
//  * m <= 8, half tiles up to 2048 rows, whose full tiles would leave half the CUs idle, where k splits
//    into 8 slices of whole batches: (2048, 2048) at 8 rows half 4.9 / full 5.7, (1024, 4096) 6.5 / 8.7; but
//    (3072, 2048) 6.7 / 6.1, (3072, 4096) 10.3 / 9.1, (4096, 4096) 10.4 / 9.5. Shared x from 5120 rows: (5120,
//    2048) shared 7.9 / full 9.1 / half 9.8, (6144, 4096) 13.4 / 15.7 / 14.5; (4096, 4096) has too few tiles.
//  * m <= 32, shared x from 8192 rows: (8192, 4096) at 16 rows 15.7 / full 18.1.
//  * k = 1024 leaves each slice one chunk and nothing to load ahead, while the full tiles' slices are one
//    batch in few registers: (8192, 1024) at 5 rows shared 6.6 / full 5.8, (12288, 1024) 8.0 / 6.9, at 12 8.7 / 8.0, at
//    24 9.3 / 10.2; (16384, 1024) at 5 9.1 / 8.4, at 16 9.7 / 10.4.
//  * m > 32: k stays whole (its LDS), so 8192 rows give shared x 128 workgroups: (8192, 2048) at 33 rows
//    shared 19.5 / full 15.0, (8192, 4096) at 48 34.2 / 31.8, at 56 34.8 / 36.1; (9216, 2048) at 33 19.8 / 23.1.
inline SkinnyForm skinny_form(int64_t rows, int64_t k, int m) {
  if (m <= 8 && rows <= 2048 && k % 2048 == 0) return kSkinnyHalf;
  bool shared;
  if (k < 2048)
    shared = rows > (m <= 8 ? 16384 : m <= 16 ? 12288 : 8192);
  else if (m <= 32)
    shared = rows >= (m <= 8 ? 5120 : 8192);
  else
    shared = rows > 8192 || (rows == 8192 && m > 48);
  return shared ? kSkinnyShared : kSkinnyFull;
}
// weight rows (and x rows of a B tile) of a tile, k per MFMA step and per batch of 4 steps, k of a
// staged chunk of x
constexpr int skinny_rows(SkinnyForm f) { return f == kSkinnyFull ? 16 : 8; }
constexpr int skinny_step(SkinnyForm f) { return f == kSkinnyFull ? 32 : 64; }
constexpr int skinny_batch(SkinnyForm f) { return 4 * skinny_step(f); }
constexpr int kSkinnyChunk = 512;

// k-slices per tile: kSkinnyWaves, a constant of the full and half kernels (known only at run time, the sum
// of the slices was a chain of LDS latencies: (2048, 1024) at 8 rows 4.3 us, so 4.1); with x shared
// 2, or 1 where 2 would only add a round of workgroups (256 CUs; (10240, 1024) at 24 rows 9.0 / 13.2) or above 32
// rows (its LDS).
inline int skinny_slices(int64_t rows, int64_t k, int m) {
  if (skinny_form(rows, k, m) != kSkinnyShared) return kSkinnyWaves;
  if (m > 32) return 1;
  const auto rounds = [&](int ks) {  // rounds of workgroups over the CUs
    const int64_t per = kSkinnyWaves / ks, wgs = (rows / 8 + per - 1) / per;
    return (wgs + 255) / 256;
  };
  return rounds(2) < 2 * rounds(1) ? 2 : 1;
}

}  // namespace kvh
