// Where the decode kernels read K in whole lines (paged_attention.hip): plain functions, also compiled for
// the host by the test that holds them to what was measured. All times in us, bf16, half-line / whole-line.
#pragma once
#include <stdint.h>

namespace kvh {

#ifndef KVH_LINE_FN
#define KVH_LINE_FN __host__ __device__ __forceinline__
#endif

// Rows of 128 bytes or more: 16-bit caches, and E4M3 caches at D = 128.
constexpr bool can_read_lines(int D, bool kv8) { return !kv8 || D == 128; }
constexpr int kLineRows = 8;  // query rows they serve

// The stream-K decode takes them for all units of a launch or for none: with both kinds on one CU the units
// ran up to 15% longer than with either kind alone (50 sequences of 2600 keys, 8 kv heads, 8 query rows, 32.0
// chunks a unit with a limit of 32 on each unit's own length: 98.2 / 112.0; one sequence in ten with 12 query
// rows among those with 4, 24 chunks a unit: 75.1 / 81.5). So the launcher looks at the bytes between K's token
// rows and at a decode-only batch's most query rows, the kernel at the mean unit and, beside prompt chunks, at
// its sequences' rows. (A cascade's prefix segments keep half lines, which other groups' reads hit in the
// caches, and its members' own keys whole ones: 4 sequences over 13000 shared keys 47.6 / 46.0.)
constexpr bool line_dim(int D) { return D == 128; }  // D = 64, one line a row: 1-4% lost in short units

// Token rows 1 to under 4 KB apart: 4, 8 or 12 kv heads of a 16-bit cache, 8, 12 or 16 of an E4M3 one. 16-bit,
// 16 chunks a unit: 8 kv heads 54.4 / 53.4, 12 56.0 / 54.2, 4 55.0 / 54.4; 16 kv heads 53.0 / 53.8, 32 2%
// slower (perhaps because rows 4 KB apart meet in one channel), 1 and 2 1-2% slower. E4M3: 8 59.2 / 58.5,
// 12 5% faster; 2, 4 and 32 1-3% slower. rows: the most query rows of a sequence (0: the kernel looks).
KVH_LINE_FN bool line_launch(int D, int rows, int64_t row_bytes) {
  return line_dim(D) && rows <= kLineRows && row_bytes >= 1024 && row_bytes < 4096;
}

// C chunks over `units` units. 16-bit caches up to 32 chunks a unit (8 kv heads 2-4% from 2 on; 4 1-3% up to 24,
// level at 32; 64 sequences of 1023-8191 keys, 73 a unit, 200.7 / 201.7); E4M3 caches from more than 8 on
// (64 sequences of 1023-8191 keys 114.9 / 113.6; 4 chunks a unit 28.7 / 29.5).
constexpr int kLineUnitChunks = 32, kLineMinChunks8 = 8;
KVH_LINE_FN bool line_units(bool kv8, int64_t C, int64_t units) {
  return kv8 ? C > kLineMinChunks8 * units : C <= kLineUnitChunks * units;
}

// The short decode, together with non-temporal loads. 16-bit caches from kShortLines = B Hkv D: 128 x 1000
// keys 102 / 88 (D = 128), 60 / 52 (D = 64), 32 x 1000 28.2 / 24.9, 16 x 500 12.4 / 11.3; below it the
// caches' half-line hits win (8 x 500 keys, D = 64: 7.3 / 8.5). E4M3 caches from kShortLines8 elements of the
// tables' K (B Hkv D W BS): 128 x 1000 keys 57.1 / 49.6 (8 kv heads), 29.5 / 27.1 (4), 131 x 300
// 39.1 / 34.0 (16), but 131 x 300 20.7 / 21.5 and 32 x 1000 16.3 / 17.8 (8). The tables may be wider than the
// keys: with 1024-token tables, from B Hkv D = 49152 up, 20-60 keys each are 0-4% faster too.
constexpr int64_t kShortLines = 16384, kShortLines8 = 48 << 20;
KVH_LINE_FN bool line_short(int D, bool kv8, int64_t rows, int64_t table_tokens) {
  return can_read_lines(D, kv8) && (kv8 ? rows * table_tokens >= kShortLines8 : rows >= kShortLines);
}

}  // namespace kvh
