// Which kernel a decode GEMV launch takes and how its sums are ordered: functions of the weight type, K, the columns and
// the number of 8-row tiles only. Host code (also compiled by itself in the tests).
#pragma once

namespace q27h {

// ggml ids of the weight types
constexpr int kQ2K = 10, kQ4K = 12, kQ6K = 14, kIQ2XXS = 16, kIQ2XS = 17, kIQ3XXS = 18, kIQ3S = 21, kIQ2S = 22,
              kIQ4XS = 23, kIQ1M = 29;

// Waves per tile, a function of the type, K and the column count only (part of the summation order). One column, and
// two for all types but IQ3_XXS / IQ3_S / IQ1_M: one block of each tile per lane, ceil(K / 2048) waves, up to K = 32768
// (16 waves); each wave adds a butterfly, which is cheap for few columns. Otherwise, and for K > 32768: at most 4 waves,
// lanes taking several blocks. Measured (us, 5120 x 17408, 4 -> 9 waves): T = 1 Q4_K 13.1 -> 10.9, IQ3_S 18.0 -> 12.5,
// IQ2_XXS 14.7 -> 9.7; T = 2 Q4_K 14.7 -> 13.5, IQ2_S 19.3 -> 14.7, but IQ3_S 15.8 -> 20.1, IQ1_M 18.1 -> 21.5; T = 4
// Q4_K 18.7 -> 25.4.
constexpr int kMaxW = 16;
constexpr int waves_per_tile(int type, int K, int ncols) {
  const int w = (K / 256 + 7) / 8;
  const bool wide = ncols == 1 || (ncols == 2 && type != kIQ3XXS && type != kIQ3S && type != kIQ1M);
  const int cap = wide ? kMaxW : 4;
  return w < 1 ? 1 : w > kMaxW ? 4 : w > cap ? cap : w;
}

// Values a launch over f32 activations may quantize per workgroup (NC * K; 40 KB of int8 in LDS).
constexpr int kFusedMaxX = 40960;

// The folding kernel (two and three columns of IQ3_XXS / IQ3_S / IQ1_M, 8192 < K <= 32768): the sums of 4 waves formed by
// one block per lane on g = ceil(K / 2048) waves. The other route has the same bits: the prefetching kernel for two
// columns, launches of two and one column for three.
constexpr bool folds(int type, int nc) { return (nc == 2 || nc == 3) && (type == kIQ3XXS || type == kIQ3S || type == kIQ1M); }
// Where the folding kernel is the faster route. It wins while workgroups are small (g <= 8: three or more on a CU, one's
// table fill, fold and reduction hidden by the others' loads) or all resident at once; a second round of large
// workgroups costs more than the waves give. us, other route -> folding:
//   two columns, 5120 x 17408 / 5120 x 10240 / 1024 x 20480: IQ3_S 16.9 / 12.0 / 9.4 -> 16.5 / 10.6 / 8.1, IQ3_XXS 16.7 /
//   11.8 / 10.1 -> 15.9 / 10.2 / 7.7, IQ1_M 18.5 / 12.9 / 11.4 -> 16.2 / 10.2 / 8.1; 17408 x 8448 IQ3_S 24.4 -> 22.5.
//   Beyond one round, other route / folding: 9..12 waves, IQ3_S x 17408: 768 tiles 1.01, 800 0.87, 896 0.77, 2176 0.81
//   (36.6 -> 45.5 us); IQ3_XXS 1.04, 0.90, 0.82, 0.85; IQ1_M never below 0.96. 13..16 waves: IQ3_S x 28672 256 tiles 1.22,
//   288 0.97, 576 0.84, x 25600 4096 tiles 0.63 (84.7 -> 134.8 us); IQ3_XXS 1.42, 1.06, 0.89, 0.67; IQ1_M 512 tiles 1.17, 576
//   0.99, 4096 0.80.
//   three columns, 5120 x 17408 / 5120 x 10240 / 1024 x 20480: IQ3_S 26.7 / 19.4 / 15.6 -> 18.5 / 11.8 / 9.3, IQ3_XXS 25.9 /
//   18.5 / 16.0 -> 18.5 / 11.6 / 9.1, IQ1_M 28.5 / 20.2 / 17.4 -> 27.8 / 13.1 / 10.8; IQ1_M alone loses: 9 waves 1280 tiles 1.02,
//   1408 0.96, 2176 0.91 (72.2 -> 78.9 us); 10..12 waves 2048 tiles 1.01-1.02, 8192 0.92-0.97.
// Four columns ran slower (5120 x 17408 Q4_K 18.6 -> 24-26, IQ3_S 20.9 -> 27.7: 9 waves of 96 VGPRs and 40 KB per
// workgroup, 640 workgroups are 1.25 rounds of the CUs).
constexpr bool fold_pays(int type, int K, int nc, int tiles) {
  const int g = (K / 256 + 7) / 8;
  if (!folds(type, nc) || g <= 4 || g > kMaxW) return false;
  if (g <= 8) return true;
  if (nc == 3) return type != kIQ1M || g > 12 || tiles <= (g == 9 ? 1280 : 2048);
  if (g <= 12) return type == kIQ1M || tiles <= 768;
  return tiles <= (type == kIQ3S ? 256 : 512);
}

// One block per lane, without prefetch registers (up to 4 waves Q2_K and Q4_K of four columns keep the prefetching kernel:
// 17408 x 5120 17.2 / 17.3 us against 18.8 / 17.9).
constexpr bool one_block(int type, int K, int nc) {
  const int w = waves_per_tile(type, K, nc == 3 ? 2 : nc);
  return K / 256 <= 8 * w && (w > 4 || !((type == kQ2K || type == kQ4K) && nc == 4));
}

// Three columns: the order of the sums is that of two columns, then that of one. One launch where both take the same waves
// (all but IQ3_XXS / IQ3_S / IQ1_M at 8192 < K <= 32768), or with the folding kernel; over f32 activations where they fit.
constexpr bool three_alike(int type, int K) { return waves_per_tile(type, K, 2) == waves_per_tile(type, K, 1); }
constexpr bool three_in_one(int type, int K, int tiles, bool fused) {
  if (fused) return three_alike(type, K) && (long)K * 3 <= kFusedMaxX;
  return three_alike(type, K) || fold_pays(type, K, 3, tiles);
}

// Whether some K takes a kernel at all; the others are not built. The prefetching kernel reads a tile's wide pieces with
// nontemporal loads up to kNtPiecesMaxK and is the only one beyond K = 32768.
constexpr int kNtPiecesMaxK = 8192;
constexpr bool one_block_reached(int type, int nc) { return one_block(type, 256, nc); }
constexpr bool prefetch_reached(int type, int nc, bool fused, bool nt) {
  for (int K = 256; K <= (fused ? kFusedMaxX / nc : 33024); K += 256)
    if (!one_block(type, K, nc) && (K <= kNtPiecesMaxK) == nt && (nc != 3 || three_alike(type, K))) return true;
  return false;
}

}  // namespace q27h
