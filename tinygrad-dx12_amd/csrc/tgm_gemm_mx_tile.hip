// The one-tile scaled-MFMA GEMM (tgm_gemm_mx_tile.h) for every FP4 / FP6 pair but E3M2 x E3M2.
#include "tgm_gemm_mx_tile.h"

namespace tgm {

// us at K = 4096 (M and N varied) for the tile shapes in launch_pair's order: FP4 x FP4, one FP6 operand, two.  The
// ratios hold down to K = 512, where the shapes that split K over waves take one or two stages, so no shape asks for a
// longest or shortest K.  The last FP4 entry is the 256 x 256 kernels' (tgm_gemm_mx.hip).
static constexpr TileCost kTiles44[] = {{32, 64, 1, 7.0f, 7.7f, 11.2f, 12.2f},    {64, 64, 1, 8.9f, 10.5f, 15.0f, 16.7f},
                                        {64, 128, 1, 10.8f, 13.2f, 23.0f, 24.8f}, {128, 128, 1, 13.7f, 18.1f, 31.0f, 34.5f},
                                        {128, 256, 1, 21.6f, 30.3f, 52.0f, 57.7f}};
static constexpr TileCost kTiles44Big[] = {kTiles44[0], kTiles44[1], kTiles44[2], kTiles44[3],
                                           {256, 256, 1, 22.5f, 39.0f, 50.0f, 78.0f}};
static constexpr TileCost kTiles64[] = {{32, 64, 1, 8.1f, 9.0f, 15.5f, 16.8f},    {64, 64, 1, 10.8f, 12.7f, 21.5f, 22.9f},
                                        {64, 128, 1, 14.8f, 17.5f, 31.0f, 34.0f}, {128, 128, 1, 17.6f, 25.0f, 41.0f, 46.7f},
                                        {128, 256, 1, 28.3f, 37.1f, 66.0f, 73.0f}};
static constexpr TileCost kTiles66[] = {{32, 64, 1, 9.4f, 10.5f, 18.5f, 20.0f},   {64, 64, 1, 13.0f, 15.0f, 25.5f, 28.0f},
                                        {64, 128, 1, 17.0f, 20.5f, 37.0f, 41.0f}, {128, 128, 1, 22.0f, 29.6f, 50.0f, 56.6f},
                                        {128, 256, 1, 36.7f, 46.0f, 83.0f, 90.0f}};

int mx_tile_shape(int ta, int tb, int64_t m, int64_t n, int64_t k, bool fp4_big, int cus) {
  const int sixes = (ta != kOpE2M1) + (tb != kOpE2M1);
  const int shape = fp4_big      ? cheapest_tile(kTiles44Big, m, n, k, cus)
                    : sixes == 0 ? cheapest_tile(kTiles44, m, n, k, cus)
                    : sixes == 1 ? cheapest_tile(kTiles64, m, n, k, cus)
                                 : cheapest_tile(kTiles66, m, n, k, cus);
  // Large products: below eight K steps gemm_f8f6f4's 256 x 128 tiles, which start and end faster, are ahead (E2M3 x
  // FP4 2048 x 4096 x 512: 12.8 against 14.4 us); from K = 1024 on the pipeline here is (K = 1152: 19.0 against 18.1).
  return shape == 4 && (fp4_big || k < 1024) ? -1 : shape;
}

template <int TA, int TB>
static int launch_pair(int shape, const MxTileArgs& p, hipStream_t s, const char* who) {
  constexpr bool both6 = F8F6F4<TA>::bits + F8F6F4<TB>::bits == 12;
  switch (shape) {
    case 0: return launch_mx_tile<TA, TB, 1, 1, 1, 2, 4, 3>(p, s, who);   // 32 x 64
    case 1: return launch_mx_tile<TA, TB, 1, 1, 2, 2, 2, 4>(p, s, who);   // 64 x 64
    case 2: return launch_mx_tile<TA, TB, 2, 1, 1, 4, 2, 3>(p, s, who);   // 64 x 128
    case 3: return launch_mx_tile<TA, TB, 2, 2, 2, 2, 2, 3>(p, s, who);   // 128 x 128
    default: return launch_mx_tile<TA, TB, 2, 2, 2, 4, 1, both6 ? 3 : 4>(p, s, who);  // 128 x 256
  }
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
