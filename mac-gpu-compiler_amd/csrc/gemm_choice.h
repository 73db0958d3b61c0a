// Which GEMM kernel and tile a launch takes, and into how many K splits: plain functions of its sizes, with
// no device code, so that a program without a GPU can ask them too.
#pragma once

#include <algorithm>
#include <cstdint>
#include <iterator>

namespace qe {

// Verify passes and chunks of up to kGemmSliceMaxM rows run the projections on k_gemm_kslice over
// f32 rows, norms and residuals within; longer chunks on k_gemm_wide over split rows.
constexpr uint32_t kGemmSliceMaxM = 64;

struct GemmTile {
  uint32_t bm, bn;
};
inline uint64_t gemm_tiles(uint64_t n, uint64_t b) { return (n + b - 1) / b; }

// ---- k_gemm_kslice ----
// (the last four: many columns, as an lm_head's, where a wide tile has fewer bytes of A beside its W)
constexpr GemmTile kSliceTiles[] = {{16, 16}, {16, 32},  {32, 32},  {32, 48},  {32, 64}, {48, 64},
                                    {64, 64}, {16, 128}, {32, 128}, {48, 128}, {64, 128}};

// The tile of a k-sliced launch: the workgroups are dealt over 256 CUs, so its time goes with the
// bytes the busiest CU loads (rounds of 256 x one workgroup's), plus what a workgroup costs besides
// its loads, worth about 60 KB of them. Measured (us, M x N x K): 9 x 6144 x 1024 on 16 x 32 tiles
// 3.5, 16 x 48 4.0; 64 x 6144 x 1024 on 32 x 48 5.8, 32 x 64 6.0, 16 x 32 7.3; 130 x 1024 x 3072 on
// 32 x 32 7.5, 32 x 64 9.0, 16 x 32 9.5; 130 x 4096 x 1024 on 48 x 64 7.3, 64 x 64 7.9, 32 x 64 10.1;
// 512 x 1024 x 3072 on 32 x 64 15.1, 48 x 64 17.6, 64 x 64 20.4. N = 151936, K = 1024 (an lm_head): 5 rows
// on 16 x 128 54.7, 64 x 128 76.5; 12 rows 56.6 and 77.9; 24 rows on 32 x 128 67.1, 64 x 128 79.7; 40 rows on
// 48 x 128 80.7, 64 x 128 84.8. Deeper rings (all of a wave's steps in flight) were slower: down of 5 rows
// 7.3 against 6.2 traced.
inline uint64_t slice_cost(uint32_t M, uint32_t N, uint32_t K, GemmTile t) {
  const uint64_t wgs = gemm_tiles(M, t.bm) * gemm_tiles(N, t.bn);
  const uint32_t rows = t.bm == 16 && M <= 8 ? 8 : t.bm;  // (HALF)
  return gemm_tiles(wgs, 256) * (uint64_t(4 * rows + 2 * t.bn) * K + 60 * 1024);
}
inline int slice_tile(uint32_t M, uint32_t N, uint32_t K) {
  int best = 0;
  for (int i = 1; i < int(std::size(kSliceTiles)); i++)
    if (slice_cost(M, N, K, kSliceTiles[i]) < slice_cost(M, N, K, kSliceTiles[best])) best = i;
  return best;
}

// ---- k_gemm_wide ----
constexpr GemmTile kWideTiles[] = {{64, 128}, {64, 192}, {128, 128}, {128, 192}, {128, 256}};

// What the tiles of a launch are ranked by: rounds of 256 workgroups, each K / 32 phases of the longer of
// its MFMAs (16 clocks each, per SIMD) and its LDS traffic (128 bytes a clock: the fragments four waves
// read and the block that is written), plus what a workgroup costs besides (fill and drain). The clocks
// are about half of those measured; the tile is the best of the five within 0.3% on average over 143
// shapes of 65 to 2048 rows (us, in the order of kWideTiles: 512 x 6144 x 1024 24.8, 18.1, 22.0, 26.7, 32.6;
// 1024 x 6144 x 1024 38.4, 34.2, 42.1, 29.6, 33.8; 2048 x 4096 x 1024 51.4, 48.7, 45.7, 52.3, 37.5), at worst
// 13% above it (700 x 8192 x 4096 119 on 64 x 192, 105 on 128 x 256).
inline uint64_t wide_cost(uint32_t M, uint32_t N, uint32_t kz, uint32_t splits, GemmTile t) {
  const uint64_t wgs = gemm_tiles(M, t.bm) * gemm_tiles(N, t.bn) * splits;
  const uint32_t mt = t.bm / 32, nt = t.bn / 32;
  const uint32_t mfma = mt * nt * 2 * 16, lds = 32 * (2 * mt + nt) + t.bm + t.bn / 2;
  return gemm_tiles(wgs, 256) * (uint64_t(kz / 32) * std::max(mfma, lds) + 7000);
}
// heads: the tile holds whole heads of 128 columns
inline GemmTile wide_tile(uint32_t M, uint32_t N, uint32_t kz, uint32_t splits, bool heads) {
  GemmTile best{};
  uint64_t cost = ~uint64_t(0);
  for (const GemmTile& t : kWideTiles) {
    if (heads && t.bn % 128) continue;
    const uint64_t c = wide_cost(M, N, kz, splits, t);
    if (c < cost) {
      cost = c;
      best = t;
    }
  }
  return best;
}

// A short K where even the largest tile makes more than one round: two workgroups a CU (rings of two slots),
// so that one writes its block while the other loads and multiplies; of 64 x 128 and 64 x 192 the one with the
// fewer columns for the busiest CU ({}: one workgroup a CU). us, one workgroup a CU / two: 2048 x 6144 x 256 27.0 /
// 22.1, x 384 32.9 / 27.3, x 96 18.7 / 16.2, 2048 x 5110 x 256 26.8 / 19.9; with 256 tiles of 128 x 256 2048 x 4096
// x 256 16.7 / 17.3.
inline GemmTile wide_pair_tile(uint32_t M, uint32_t N, uint32_t K) {
  if (K > 512 || gemm_tiles(M, 128) * gemm_tiles(N, 256) <= 256) return {};
  const uint64_t rows = gemm_tiles(M, 64);
  const bool narrow = gemm_tiles(rows * gemm_tiles(N, 128), 256) * 128 < gemm_tiles(rows * gemm_tiles(N, 192), 256) * 192;
  return narrow ? GemmTile{64, 128} : GemmTile{64, 192};
}

// A plain product of f32 rows (qe_op_gemm_bf16): on k_gemm_wide, or on k_gemm_kslice.
// More than 64 rows: the k-sliced kernel while its largest tile makes one round of 256 workgroups (us, it and
// the wide one, each on its own tile: 130 x 6144 x 1024 9.5 and 12.8, 333 x 4096 x 1024 11.1 and 13.0; past it
// 512 x 6144 x 1024 24.2 and 18.1, 333 x 6144 x 1024 18.8 and 16.2), but its two largest tiles only over a K that
// makes up for their sums through LDS (48 x 128: K = 320 8.0 and 7.2, 1024 11.2 and 13.2; 64 x 128: 96 6.7 and
// 5.5, 1024 17.1 and 15.3, 1664 21.5 and 19.7, 2048 26.7 and 28.3, 3040 30.4 and 34.4).
inline bool gemm_on_wide(uint32_t M, uint32_t N, uint32_t K) {
  if (M <= kGemmSliceMaxM) return false;
  if (gemm_tiles(M, 64) * gemm_tiles(N, 128) > 256) return true;
  const GemmTile t = kSliceTiles[slice_tile(M, N, K)];
  const uint32_t area = t.bm * t.bn;
  return K < (area >= 64 * 128 ? 2048u : area >= 48 * 128 ? 672u : 0u);
}

// ---- a chunk ----
// Whether a chunk of M rows takes split rows and k_gemm_wide (H, I: hidden and intermediate size). At widths
// that are no multiple of 64 that is from 320 tiles of 64 x 128 of gate|up (prefill, us, k_gemm_kslice / split
// rows: hidden 1056 / intermediate 3104 350 tokens 818 / 889, 400 912 / 918, 450 939 / 867; 544 / 1568 600 566 /
// 617, 800 720 / 669; 2080 / 4064 256 509 / 579, 350 625 / 620, 400 720 / 656; 1056 / 3104 in one chunk of 2048 4180 /
// 2380), otherwise from 65 rows (1024 / 3072, 28 layers: 200 tokens 1927 / 1841, 256 2063 / 1952, 333 2543 / 2244;
// below that the other way round, 65 1429 / 1653, 100 1545 / 1743, 130 1751 / 1786: one more block of 64 rows would
// pay on k_gemm_kslice).
inline bool chunk_on_split_rows(uint32_t M, uint32_t H, uint32_t I) {
  if (M <= kGemmSliceMaxM || H % 32 || I % 32) return false;
  return (H % 64 == 0 && I % 64 == 0) || gemm_tiles(M, 64) * gemm_tiles(2 * uint64_t(I), 128) > 320;
}

// K splits for launch_gemm_split: 64 x 128 tiles, split while that leaves CUs without one (1 when K does not
// split)
inline uint32_t gemm_splits(uint32_t M, uint32_t N, uint32_t K) {
  const uint64_t tiles = gemm_tiles(N, 128) * gemm_tiles(M, 64);
  uint32_t z = 1;
  while (z < 8 && tiles * z < 256 && K % (128 * z) == 0) z *= 2;
  return z;
}

}  // namespace qe
