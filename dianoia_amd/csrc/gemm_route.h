// Which kernel dnx_gemm_q8 / dnx_gemm_q4 (gemm.hip) run for a shape, and into
// how many parts the tile kernel splits K. Host code alone, without HIP.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace dnx {

enum class GemmKernel {
  kSkinny,          // up to 16 tokens: 16 weight rows a workgroup, one launch
  kChunk1, kChunk2, // a prompt chunk: 32 rows x 32 or 64 tokens, one launch
  kTile32, kTile64, // 32 x 128 or 64 x 64 tiles, K split where they are few
};

// LDS of the skinny kernel: padded weight rows, weight scales (fp32), x
// scales [block][token], and waves 1..3's sums.
constexpr int kSkinnyRows = 16;
inline size_t skinny_lds(bool q4, int64_t cols, int mt) {
  const size_t blocks = (size_t)cols / 32, row = (size_t)(q4 ? cols / 2 : cols) + 16;
  return kSkinnyRows * row + kSkinnyRows * blocks * 4 + blocks * 16 * mt * 4 +
         (size_t)3 * mt * 4 * 64 * 4;
}

// Whether the skinny kernel takes this shape: n <= 16, K <= 2048 (16
// blocks per wave, 8 row pieces per thread) and the LDS within 64 KB. With
// more tokens it lost to the split-K tile kernel on 6144 x 2048 Q4 (n = 32:
// 13.7 against 11.8 us; n = 16: 9.7 against 10.2; n = 8: 8.5 against 9.4).
inline bool skinny_fits(bool q4, int64_t cols, int64_t n) {
  return n <= 16 && cols <= 2048 && skinny_lds(q4, cols, 1) <= 64 * 1024;
}

// Token groups per workgroup of the chunk kernel for a shape, 0 where the
// tile kernel is the faster (graph-timed with the quantizer, us, tile kernel
// against this):
// * one round of 256 workgroups, or the second round's tail costs more than
//   the tile kernel's reduce (3072 x 1024 at 200 tokens: 14.6 against 14.4,
//   6144 x 1024 at 200 14.9 against 20.0);
// * K <= 1024 (a wave's blocks all requested at once): Q8 3072 x 1024 at 33 /
//   64 / 128 tokens 9.2 / 10.8 / 12.2 against 7.2 / 7.3 / 9.0, Q4 9.2 / 10.9 /
//   12.0 against 7.8 / 7.9 / 9.7, 512 x 512 at 17..256 7.7..8.5 against 5.7..6.3;
// * K <= 2048 (two units a wave) where the launch fills the chip enough: 2048
//   x 2048 Q8 at 64 / 128 12.8 / 13.7 against 10.2 / 10.4, Q4 12.5 / 13.6
//   against 11.4 / 11.9; with 64 workgroups or fewer (512 x 2048 Q8 at 64: 9.0
//   against 9.9), and below 64 tokens of Q4 (2048 x 2048 at 33: 10.1 against
//   11.3), the tile kernel's K split wins;
// * longer K: each unit adds a memory round trip (1024 x 3072 at 64: 11.7
//   against 12.9);
// * K <= 128 is one stage of the tile kernel, which then needs no reduce
//   either, and one unit, so that one wave in eight multiplies (the products
//   alone): it stays with the tile kernel but for one token group and up to 96
//   (916 x 32 at 58 3.4 against 3.1, 1342 x 96 at 81 3.7 against 3.3; 2118 x
//   128 at 60 3.8 against 4.0, 79 x 128 at 373 3.8 against 4.0; two groups:
//   2941 x 32 at 121 3.5 against 3.8, 1899 x 96 Q4 at 131 3.8 against 4.1).
// Up to 16 tokens the skinny kernel's sums are closer to 64 bits (7.2e-8
// against 8.4e-8 at K = 1024) and it keeps them.
inline int chunk_groups(bool q4, int64_t rows, int64_t cols, int64_t n) {
  const int64_t blocks = cols / 32, row_groups = (rows + 31) / 32;
  if (n <= 16 || blocks > 64 || blocks == 4) return 0;
  for (int g = 1; g <= 2; g++) {
    const int64_t wgs = row_groups * ((n + 32 * g - 1) / (32 * g));
    if (wgs > 256) continue;
    if (blocks < 4) return g == 1 ? 1 : 0;
    return blocks <= 32 || (wgs > 64 && (!q4 || n >= 64)) ? g : 0;
  }
  return 0;
}

// 32 tokens: one wave row of 32 x 32 tiles (4 waves across N); else 64 x 64
// tiles (2 x 2 waves), which keep ~3 workgroups per CU resident at prefill
// sizes.
inline GemmKernel gemm_kernel_for(bool q4, int64_t rows, int64_t cols, int64_t n) {
  if (skinny_fits(q4, cols, n)) return GemmKernel::kSkinny;
  const int groups = chunk_groups(q4, rows, cols, n);
  if (groups > 0) return groups == 1 ? GemmKernel::kChunk1 : GemmKernel::kChunk2;
  return n <= 32 ? GemmKernel::kTile32 : GemmKernel::kTile64;
}

// Stages of K (4 blocks each) that a workgroup of the tile kernel takes.
// K is split when the tiles alone would leave CUs idle (small n): enough
// splits for about 512 workgroups, each with at least one stage. Between
// one and three workgroups per CU (the resident count of the 64 x 64
// tiles) a long K (32+ stages) is split too, into runs of at least 8
// stages, so that the slots fill: the vision fc2 (1152 x 4320 at 1024
// tokens, 288 tiles) ran one or two workgroups per CU over all 34 stages
// (47.9 -> 42.6 us with 3 splits). A shorter K loses more to the partials'
// round trip than it gains (6144 x 2048 at 256 tokens: 24 -> 27 us).
constexpr int kTileBlocks = 4;
inline int tile_split_stages(int64_t tiles, int stages) {
  int splits = 1;
  if (tiles < 256 && stages > 1) {
    splits = (int)((512 + tiles - 1) / tiles);
    if (splits > stages) splits = stages;
  } else if (tiles < 768 && stages >= 32) {
    splits = (int)((768 + tiles - 1) / tiles);
    if (splits > stages / 8) splits = stages / 8;
  }
  return (stages + splits - 1) / splits;
}

}  // namespace dnx
