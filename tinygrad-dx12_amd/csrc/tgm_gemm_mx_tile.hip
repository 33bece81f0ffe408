// The one-tile scaled-MFMA GEMM (tgm_gemm_mx_tile.h) for every FP4 / FP6 pair but E3M2 x E3M2.
#include "tgm_gemm_mx_tile.h"

namespace tgm {

// us at K = 4096 (M and N varied) for the tile shapes in launch_pair's order, then for the kernel of large
// tiles that competes with them: gemm_f8f6f4's 256 x 128 (one workgroup per tile, two on a compute unit for FP4
// x FP4), and the 256 x 256 kernels of tgm_gemm_mx.hip for FP4 pairs that they take.  gemm_f8f6f4 starts and
// ends faster and falls behind with K, so its tables know what does not grow with K (measured at K = 384 to
// 7552).  FP4 x FP4, one FP6 operand, two:
//   1348 x 14336 x 640, FP4 x FP4: 19.7 us, 27.0 on 128 x 256 tiles; 3000 x 14336 x 2432: 80.2 against 107.6
//   4096 x 9842 x 1152, E2M3 x FP4: 149 against 161 us; 2048 x 4096 x 7552: 66 against 58
// FP4 x FP4 has no 128 x 256 entry: at its best (3/4 to one round, K >= 4224) it is 10 to 20 % ahead of 256 x
// 128, at shorter K and in other rounds up to 65 % behind.
static constexpr TileCost kTiles44[] = {{32, 64, 1, 7.0f, 7.7f, 11.2f, 12.2f, 0.38f},
                                        {64, 64, 1, 8.9f, 10.5f, 15.0f, 16.7f, 0.34f},
                                        {64, 128, 1, 10.8f, 13.2f, 23.0f, 24.8f, 0.34f},
                                        {128, 128, 1, 13.7f, 18.1f, 31.0f, 34.5f, 0.35f},
                                        {256, 128, 1, 18.8f, 30.0f, 34.5f, 46.0f, 0.19f}};
static constexpr TileCost kTiles44Big[] = {{32, 64, 1, 7.0f, 7.7f, 11.2f, 12.2f},    {64, 64, 1, 8.9f, 10.5f, 15.0f, 16.7f},
                                           {64, 128, 1, 10.8f, 13.2f, 23.0f, 24.8f}, {128, 128, 1, 13.7f, 18.1f, 31.0f, 34.5f},
                                           {256, 256, 1, 22.5f, 39.0f, 50.0f, 78.0f}};
static constexpr TileCost kTiles64[] = {{32, 64, 1, 8.1f, 9.0f, 15.5f, 16.8f, 0.43f},
                                        {64, 64, 1, 10.8f, 12.7f, 21.5f, 22.9f, 0.36f},
                                        {64, 128, 1, 14.8f, 17.5f, 31.0f, 34.0f, 0.30f},
                                        {128, 128, 1, 17.6f, 25.0f, 41.0f, 46.7f, 0.32f},
                                        {128, 256, 1, 28.3f, 37.1f, 66.0f, 73.0f, 0.235f},
                                        {256, 128, 1, 31.0f, 39.2f, 67.0f, 74.0f, 0.165f}};
static constexpr TileCost kTiles66[] = {{32, 64, 1, 9.4f, 10.5f, 18.5f, 20.0f, 0.41f},
                                        {64, 64, 1, 13.0f, 15.0f, 25.5f, 28.0f, 0.31f},
                                        {64, 128, 1, 17.0f, 20.5f, 37.0f, 41.0f, 0.29f},
                                        {128, 128, 1, 22.0f, 29.6f, 50.0f, 56.6f, 0.31f},
                                        {128, 256, 1, 36.7f, 46.0f, 83.0f, 90.0f, 0.18f},
                                        {256, 128, 1, 41.2f, 49.2f, 87.0f, 91.0f, 0.13f}};
static constexpr int kGroups[] = {4, 2, 2, 2, 1};  // launch_pair's K groups by shape

template <int COUNT>
static int choose(const TileCost (&table)[COUNT], int64_t m, int64_t n, int64_t k, int cus, TileChoice* tile) {
  const int i = cheapest_tile(table, m, n, k, cus);
  const bool large = i == COUNT - 1;
  if (tile) *tile = {table[i].bm, table[i].bn, large ? 1 : kGroups[i], large ? kLargeTile : kOneTile};
  return large ? -1 : i;
}

int mx_tile_shape(int ta, int tb, int64_t m, int64_t n, int64_t k, bool fp4_big, int cus, TileChoice* tile) {
  if (fp4_big) return choose(kTiles44Big, m, n, k, cus, tile);
  switch ((ta != kOpE2M1) + (tb != kOpE2M1)) {
    case 0: return choose(kTiles44, m, n, k, cus, tile);
    case 1: return choose(kTiles64, m, n, k, cus, tile);
    default: return choose(kTiles66, m, n, k, cus, tile);
  }
}

template <int TA, int TB>
static int launch_pair(int shape, const MxTileArgs& p, hipStream_t s, const char* who) {
  constexpr int sixes = (TA != kOpE2M1) + (TB != kOpE2M1);
  switch (shape) {
    case 0: return launch_mx_tile<TA, TB, 1, 1, 1, 2, 4, 3>(p, s, who);   // 32 x 64
    case 1: return launch_mx_tile<TA, TB, 1, 1, 2, 2, 2, 4>(p, s, who);   // 64 x 64
    case 2: return launch_mx_tile<TA, TB, 2, 1, 1, 4, 2, 3>(p, s, who);   // 64 x 128
    case 3: return launch_mx_tile<TA, TB, 2, 2, 2, 2, 2, 3>(p, s, who);   // 128 x 128
    default: break;
  }
  if constexpr (sixes > 0) return launch_mx_tile<TA, TB, 2, 2, 2, 4, 1, sixes == 2 ? 3 : 4>(p, s, who);  // 128 x 256
  TGM_UNSUPPORTED("%s: no tile shape %d", who, shape);
}

int launch_gemm_mx_tile(int shape, int ta, int tb, const MxTileArgs& p, hipStream_t s, const char* who) {
#define TGM_MX_PAIR(A, B) \
  if (ta == A && tb == B) return launch_pair<A, B>(shape, p, s, who);
  TGM_MX_PAIR(kOpE2M1, kOpE2M1) TGM_MX_PAIR(kOpE2M1, kOpE2M3) TGM_MX_PAIR(kOpE2M1, kOpE3M2)
  TGM_MX_PAIR(kOpE2M3, kOpE2M1) TGM_MX_PAIR(kOpE2M3, kOpE2M3) TGM_MX_PAIR(kOpE2M3, kOpE3M2)
  TGM_MX_PAIR(kOpE3M2, kOpE2M1) TGM_MX_PAIR(kOpE3M2, kOpE2M3)
#undef TGM_MX_PAIR
  TGM_UNSUPPORTED("%s: no scaled-MFMA kernel for operand types %d x %d", who, ta, tb);
}

}  // namespace tgm
