// The one-tile weight GEMM (tgm_gemm_w_tile.h) for FP4 and FP6 weights.
#include "tgm_gemm_w_tile.h"

namespace tgm {

// us at K = 4096 (N and M varied), FP4 / FP6 E2M3.  The 32 x 64 shape needs 50 KB of LDS per stage for FP6.
// FP6 knows the share that does not grow with K: smaller tiles have more of it (E3M2 700 x 14336 x 128: 16.9 us on
// 128 x 128, 14.8 on 128 x 256).
static constexpr TileCost kFp4Tiles[] = {
    {32, 32, 4, 7.1f, 8.7f, 14.4f, 16.0f},   {32, 64, 4, 8.5f, 10.5f, 18.3f, 19.0f},  {64, 64, 2, 11.4f, 14.4f, 24.5f, 27.0f},
    {64, 128, 1, 17.7f, 21.5f, 31.4f, 38.4f}, {128, 128, 1, 26.7f, 34.2f, 60.0f, 67.0f}, {128, 256, 1, 38.6f, 53.0f, 94.0f, 106.0f}};
static constexpr TileCost kFp6Tiles[] = {{32, 32, 4, 7.3f, 9.3f, 16.0f, 17.6f, 0.15f},
                                         {64, 64, 2, 11.4f, 16.1f, 26.5f, 31.6f, 0.15f},
                                         {64, 128, 1, 17.7f, 25.5f, 41.5f, 47.0f, 0.15f},
                                         {128, 128, 1, 27.0f, 35.6f, 60.0f, 73.0f, 0.15f},
                                         {128, 256, 1, 48.0f, 58.4f, 106.0f, 117.0f, 0.11f}};

TileChoice w_tile_mx(int fmt, int64_t m, int64_t n, int64_t k, int cus) {
  const TileCost& t = fmt == TGM_FMT_FP4_E2M1 ? kFp4Tiles[cheapest_tile(kFp4Tiles, m, n, k, cus)]
                                              : kFp6Tiles[cheapest_tile(kFp6Tiles, m, n, k, cus)];
  return {t.bm, t.bn, t.wk, kOneTile};
}

int launch_gemm_w_tile_mx(const WTileArgs& p, int fmt, int cus, hipStream_t st) {
  if (fmt == TGM_FMT_FP4_E2M1) {
    constexpr int F = TGM_FMT_FP4_E2M1;
    switch (cheapest_tile(kFp4Tiles, p.M, p.N, p.K, cus)) {
      case 0: return launch_w_tile<F, 1, 1, 4, 3>(p, 1, st);
      case 1: return launch_w_tile<F, 1, 2, 4, 3>(p, 1, st);
      case 2: return launch_w_tile<F, 2, 2, 2, 3>(p, 1, st);
      case 3: return launch_w_tile<F, 2, 4, 1, 3>(p, 1, st);
      case 4: return launch_w_tile<F, 4, 4, 1, 3>(p, 1, st);
      default: return launch_w_tile<F, 4, 8, 1, 3>(p, 1, st);
    }
  }
  const int shape = cheapest_tile(kFp6Tiles, p.M, p.N, p.K, cus);
#define TGM_FP6_TILES(F)                                     \
  switch (shape) {                                           \
    case 0: return launch_w_tile<F, 1, 1, 4, 3>(p, 1, st);   \
    case 1: return launch_w_tile<F, 2, 2, 2, 3>(p, 1, st);   \
    case 2: return launch_w_tile<F, 2, 4, 1, 3>(p, 1, st);   \
    case 3: return launch_w_tile<F, 4, 4, 1, 3>(p, 1, st);   \
    default: return launch_w_tile<F, 4, 8, 1, 2>(p, 1, st);  \
  }
  if (fmt == TGM_FMT_FP6_E2M3) {
    TGM_FP6_TILES(TGM_FMT_FP6_E2M3)
  }
  TGM_FP6_TILES(TGM_FMT_FP6_E3M2)
#undef TGM_FP6_TILES
}

}  // namespace tgm
