// The main loop of the skinny GEMMs (up to 64 rows of x against a weight streamed once): one
// wave's k-slice of a weight tile on v_mfma_f32_16x16x32. HBM-bound on the weight; three forms
// keep HBM busy over the range of shapes (times on (n, k), cold weights, bf16):
//
//  kSkinnyFull    16 weight rows as the A operand, a load reading 64 bytes of each, 16 rows of x
//                 per B tile straight from the caches; k split over 8 waves. Weights of few rows.
//  kSkinnyHalf    m <= 8: the A operand is 8 weight rows twice, rows i and i + 8 the same row at
//                 two neighbouring 8-element chunks, and the B operand 8 rows of x likewise: the
//                 products of equal halves sum to the result, those of unequal ones are dropped.
//                 A load then reads whole 128-byte lines of 8 rows, non-temporally (nothing reads
//                 the weight again in this step), and twice the tiles fill the chip: (2048, 8192)
//                 at 8 rows 14.6 -> 10.4 us, (2048, 2048) 5.7 -> 4.9.
//  kSkinnyShared  the half tiles for any m, ceil(m / 8) B tiles, with x staged in LDS in chunks,
//                 one chunk ahead, and shared by the workgroup's tiles. Read from the caches by
//                 every wave, x took the L1's bandwidth from the weight: (128256, 4096) 240 us at
//                 8 rows and 399 at 32, against 185 and 219 with x left out. For weights of many
//                 rows, whose tiles fill the chip with k split little.
#pragma once

#include <type_traits>

#include "kvh_device.h"
#include "skinny_form.h"

namespace kvh {

// LDS of a workgroup: x's chunks of all slices twice (each row padded so that the rows of an
// operand read fall on different banks), or the partial tiles at the end.
constexpr int kSkinnyRowBytes = 2 * kSkinnyChunk + 32;
template <SkinnyForm F, int MT>
constexpr int skinny_lds_bytes(int ks) {
  const int xs = F == kSkinnyShared ? 2 * ks * 8 * MT * kSkinnyRowBytes : 0, red = kSkinnyWaves * MT * 64 * 16;
  return xs > red ? xs : red;
}

// This lane's place in an operand: its row of the tile (of 8 or 16) and the offset of its first 8
// elements of k.
template <SkinnyForm F>
__device__ __forceinline__ int skinny_row(int lane) {
  return F == kSkinnyFull ? lane & 15 : lane & 7;
}
template <SkinnyForm F>
__device__ __forceinline__ int skinny_k(int lane) {
  return F == kSkinnyFull ? 8 * (lane >> 4) : 16 * (lane >> 4) + (lane & 8);
}

// acc[t] += (x rows of B tile t) . (the tile's weight rows) over slice `slice` of the
// workgroup's ks, `len` of k (whole batches, or chunks). wr: this lane's first elements of the
// weight; x, x_rs, m: the rows of x (past m, row m - 1 is read); lds: skinny_lds_bytes.
// ONE: a slice is one batch (full tiles at k = 1024), with no second set of registers: 38 instead of 82 at
// 16 rows of x, so the workgroups of up to 16384 weight rows fit the chip at once ((12288, 1024) at 5 rows 8.9 us,
// so 6.9).
template <class E, SkinnyForm F, int MT, bool ONE>
__device__ __forceinline__ void skinny_slice(const uint16_t* wr, const uint16_t* x, int64_t x_rs, int m, int ks,
                                             int slice, int len, char* lds, f32x4 (&acc)[MT]) {
  constexpr int U = 4, STEP = skinny_step(F), BATCH = skinny_batch(F), ROWS = skinny_rows(F) * MT;
  const int lane = threadIdx.x & 63;
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  u32x4 a[ONE ? 1 : 2][U];
  auto load_a = [&](auto S, int kk) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const u32x4* src = (const u32x4*)(wr + kk + STEP * u);
      if constexpr (F == kSkinnyFull)
        a[decltype(S)::value][u] = *src;  // half lines: the other half is read from the cache
      else
        a[decltype(S)::value][u] = __builtin_nontemporal_load(src);
    }
  };
  auto mfmas = [&](auto S, const u32x4 (&b)[U][MT]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = E::mfma(a[decltype(S)::value][u], b[u][t], acc[t]);
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (F != kSkinnyShared) {
    const uint16_t* xr[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
      xr[t] = x + (int64_t)min(skinny_rows(F) * t + skinny_row<F>(lane), m - 1) * x_rs + slice * len + skinny_k<F>(lane);
    u32x4 b[ONE ? 1 : 2][U][MT];
    auto load = [&](auto S, int kk) {
      load_a(S, kk);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t) b[decltype(S)::value][u][t] = *(const u32x4*)(xr[t] + kk + STEP * u);
      __builtin_amdgcn_sched_barrier(0);
    };
    load(S0{}, 0);
    if constexpr (ONE) {
      mfmas(S0{}, b[0]);
    } else {
      int kk = 0;
      for (; kk + 2 * BATCH < len; kk += 2 * BATCH) {
        load(S1{}, kk + BATCH);
        mfmas(S0{}, b[0]);
        load(S0{}, kk + 2 * BATCH);
        mfmas(S1{}, b[1]);
      }
      if (kk + BATCH < len) {
        load(S1{}, kk + BATCH);
        mfmas(S0{}, b[0]);
        mfmas(S1{}, b[1]);
      } else {
        mfmas(S0{}, b[0]);
      }
    }
  } else {
    constexpr int VPR = kSkinnyChunk / 8, THREADS = 64 * kSkinnyWaves;
    constexpr int VT = 2 * ROWS * VPR / THREADS;  // 16-byte vectors per thread at ks = 2
    static_assert(kSkinnyChunk == 2 * BATCH && ROWS * VPR % THREADS == 0, "a chunk is two batches");
    u32x4 xv[VT];
    // vector q of a chunk: slice q / (ROWS VPR), row q / VPR % ROWS, k 8 (q % VPR)
    const int nv = ks * ROWS * VPR;
    auto x_load = [&](int kk) {
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        const int q = threadIdx.x + THREADS * v;
        if (THREADS * v >= nv) continue;  // uniform
        const int r = q / VPR % ROWS;
        xv[v] = *(const u32x4*)(x + (int64_t)min(r, m - 1) * x_rs + (int64_t)(q / (ROWS * VPR)) * len + kk + 8 * (q % VPR));
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto x_store = [&](int buf) {
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        const int q = threadIdx.x + THREADS * v;
        if (THREADS * v >= nv) continue;
        *(u32x4*)(lds + (buf * ks * ROWS + q / VPR) * kSkinnyRowBytes + 16 * (q % VPR)) = xv[v];
      }
    };
    const int rd = (slice * ROWS + skinny_row<F>(lane)) * kSkinnyRowBytes + 2 * skinny_k<F>(lane);
    auto mma = [&](auto S, int buf) {
      const char* src = lds + buf * ks * ROWS * kSkinnyRowBytes + rd + decltype(S)::value * BATCH * 2;
      u32x4 b[U][MT];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t) b[u][t] = *(const u32x4*)(src + 8 * t * kSkinnyRowBytes + 2 * STEP * u);
      mfmas(S, b);
    };
    load_a(S0{}, 0);
    __builtin_amdgcn_sched_barrier(0);
    x_load(0);
    x_store(0);
    __syncthreads();
    // every load is unconditional: past the end the last chunk's x and batch are read again
    for (int kk = 0, buf = 0; kk < len; kk += kSkinnyChunk, buf ^= 1) {
      load_a(S1{}, kk + BATCH);
      __builtin_amdgcn_sched_barrier(0);
      x_load(min(kk + kSkinnyChunk, len - kSkinnyChunk));
      mma(S0{}, buf);
      load_a(S0{}, min(kk + kSkinnyChunk, len - BATCH));
      __builtin_amdgcn_sched_barrier(0);
      mma(S1{}, buf);
      x_store(buf ^ 1);  // last read before the previous barrier
      __syncthreads();
    }
  }
}

// The sums of lane l (4 weight rows 4 (l / 16) .. of a tile, x row l % 16 of B tile t) over the
// tile's ks slices, in slice order. Half tiles: l % 16 < 8 and l < 32, the other half's sums
// being those of lane l + 40 (rows + 8, columns + 8).
template <SkinnyForm F, int MT>
__device__ __forceinline__ f32x4 skinny_sum(const f32x4 (*red)[MT][64], int ks, int t, int l) {
  f32x4 o = red[0][t][l];
  if constexpr (F != kSkinnyFull) o += red[0][t][l + 40];
#pragma unroll
  for (int v = 1; v < (F == kSkinnyShared ? 2 : kSkinnyWaves); ++v) {
    if (v >= ks) break;
    o += red[v][t][l];
    if constexpr (F != kSkinnyFull) o += red[v][t][l + 40];
  }
  return o;
}

}  // namespace kvh
