// gemm_choice.h -- which tile a GEMM takes, from its sizes alone (host code).
#pragma once

#include <cstdint>
#include <initializer_list>

namespace rgnpu {

// Tile shape of the large GEMM: 256, 192 or 128 rows x 256 columns (8 waves), or
// 128 x 128 (4 waves); splits > 1 when K is split.  The tiles of M rows cover no
// more than Mpad.
struct GemmChoice {
  int bm, bn;
  int splits;
};

// Kernel choice.  Problems with at least 256 tiles of 256 x 128 take 256
// columns and the number of rows (256, 192 or 128) whose rounds of one workgroup
// per CU take the least time: a K step of a tile takes bm + 104 parts (one
// round of 256 tiles, K = 4096 INT8: 54.3, 44.2 and 34.8 us; FP16 of the same
// bytes x 2: 105, 83.3 and 64.5 us), so 3000 x 4096 runs as 256 tiles of 192 rows in
// one round, where 384 tiles of 256 x 128 left half the CUs idle for the second
// half (FP16, K 4096: 151 -> 113 us a layer).  A last round of part of the CUs
// takes 0.6 of a round and 0.4 of its share (clock and memory are shared by fewer):
// 8192 x 2000 x 3000 is 384 tiles of 256 rows, 77 us with the next layer's
// quantization, rather than 3 full rounds of 128 rows, 85; 5100 x 4096 x 4096 320,
// 113 us against 123.  Over 192 shapes the choice was the fastest or within 5%.
// Smaller problems use 128 x 128 tiles and, below 128 tiles (fewer than half the
// CUs busy), split K over up to 512 blocks of at least 4 K steps each through the
// workspace.
inline GemmChoice choose_gemm(int64_t M, int64_t Mpad, int64_t Npad, int64_t Kpad) {
  if (Mpad % 256 == 0 && Npad % 256 == 0 && (Mpad / 256) * (Npad / 128) >= 256) {
    int best = 0;
    int64_t best_cost = 0;
    for (int bm : {256, 192, 128}) {
      const int64_t tiles_m = (M + bm - 1) / bm;
      if (tiles_m * bm > Mpad) continue;
      const int64_t tiles = tiles_m * (Npad / 256), part = tiles % 256;
      const int64_t cost = (bm + 104) * (tiles / 256 * 1280 + (part ? 768 + 2 * part : 0));
      if (!best || cost < best_cost) {
        best = bm;
        best_cost = cost;
      }
    }
    return {best, 256, 1};
  }
  const int64_t tiles = (Mpad / 128) * (Npad / 128), nk = Kpad / 64;
  if (tiles >= 128) return {128, 128, 1};
  int64_t S = 512 / (tiles > 0 ? tiles : 1);
  if (S > nk / 4) S = nk / 4;
  if (S < 1) S = 1;
  const int64_t ks = (nk + S - 1) / S;
  return {128, 128, (int)((nk + ks - 1) / ks)};
}

// Estimated time of launch_gemm_f32 in us.  The matrix cores take 1.0 us per K
// step (64 bytes of each row) of a 128 x 128 tile and 5 us around it, a tile per
// CU and round; split sums go through memory and a second kernel (777 x 4096 x
// 4096 estimated 265, measured 272; 200 x 4096 x 4096, K in 8 slices, 84 and 82;
// 1300 x 1024 x 8192 211 and 211).
inline double gemm_f32_us(int64_t M, int64_t Mpad, int64_t Npad, int64_t Kpad_bytes) {
  const GemmChoice g = choose_gemm(M, Mpad, Npad, Kpad_bytes);
  const int64_t nk = Kpad_bytes / 64;
  if (g.splits > 1) {
    const int64_t rounds = ((Mpad / 128) * (Npad / 128) * g.splits + 255) / 256;
    return 7.0 + (double)(rounds * ((nk + g.splits - 1) / g.splits)) + (double)(g.splits * Mpad * Npad) * 8.0 / 5e6;
  }
  const int64_t rounds = ((M + g.bm - 1) / g.bm * (Npad / g.bn) + 255) / 256;
  return 4.0 + (double)rounds * (double)(g.bm * g.bn) / 16384.0 * (double)(nk + 5);
}

}  // namespace rgnpu
