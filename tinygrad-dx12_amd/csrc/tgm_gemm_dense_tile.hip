// The one-tile bf16 / f16 GEMM (tgm_gemm_dense_tile.h).
#include "tgm_gemm_dense_tile.h"

namespace tgm {

// us at K = 4096 (M and N varied) for the shapes in launch_dtype's order; the ratios hold from K = 512 to 8192, so no
// shape asks for a longest or shortest K.  Below, the smaller tiles' larger share that does not grow with K counts
// (700 x 14336 x 128: 16.0 us on 128 x 128, 14.5 on 128 x 256).
static constexpr TileCost kDenseTiles[] = {{32, 64, 1, 10.2f, 13.2f, 21.0f, 24.0f, 0.15f},
                                           {64, 64, 1, 12.5f, 16.2f, 28.0f, 30.7f, 0.15f},
                                           {64, 128, 1, 17.0f, 24.0f, 39.0f, 43.2f, 0.15f},
                                           {128, 128, 1, 26.5f, 34.8f, 60.0f, 67.5f, 0.15f},
                                           {128, 256, 1, 43.3f, 62.0f, 98.0f, 118.0f, 0.11f}};
static constexpr int kGroups[] = {4, 2, 2, 1, 1};  // launch_dtype's K groups by shape

int dense_tile_shape(int64_t m, int64_t n, int64_t k, int cus, TileChoice* tile) {
  const int i = cheapest_tile(kDenseTiles, m, n, k, cus);
  if (tile) *tile = {kDenseTiles[i].bm, kDenseTiles[i].bn, kGroups[i], kOneTile};
  return i;
}

template <int T16>
static int launch_dtype(int shape, const DenseTileArgs& p, hipStream_t s) {
  switch (shape) {
    case 0: return launch_dense_tile<T16, 1, 1, 1, 2, 4, 3>(p, s);   // 32 x 64
    case 1: return launch_dense_tile<T16, 1, 1, 2, 2, 2, 4>(p, s);   // 64 x 64
    case 2: return launch_dense_tile<T16, 2, 1, 1, 4, 2, 3>(p, s);   // 64 x 128
    case 3: return launch_dense_tile<T16, 2, 2, 2, 2, 1, 4>(p, s);   // 128 x 128
    default: return launch_dense_tile<T16, 2, 2, 2, 4, 1, 3>(p, s);  // 128 x 256
  }
}

int launch_gemm_dense_tile(int shape, int dtype, const DenseTileArgs& p, hipStream_t s) {
  return dtype == TGM_BF16 ? launch_dtype<TGM_BF16>(shape, p, s) : launch_dtype<TGM_F16>(shape, p, s);
}

}  // namespace tgm
