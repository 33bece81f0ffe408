// The one-tile weight GEMM (tgm_gemm_w_tile.h) for INT4 / UINT4 weights with f16, bf16 or fp32 scales.
#include "tgm_gemm_w_tile.h"

namespace tgm {

// us at K = 4096 with fp16 scales per 128 and per 32 (every 32 K-elements the partial sums cost FA x 16 FMAs
// per wave, so the small tiles pay more for them).
static constexpr TileCost kI4Tiles[] = {
    {32, 32, 4, 9.0f, 10.3f, 17.5f, 18.1f},   {32, 64, 4, 9.8f, 11.3f, 19.9f, 22.3f},   {64, 64, 2, 15.9f, 18.6f, 32.0f, 33.6f},
    {64, 128, 2, 21.3f, 25.1f, 43.0f, 48.0f}, {64, 128, 1, 23.6f, 28.5f, 36.0f, 43.4f}, {128, 256, 1, 48.0f, 67.6f, 111.0f, 120.0f}};
static constexpr TileCost kI4Tiles32[] = {
    {32, 32, 4, 12.2f, 13.8f, 24.4f, 25.5f},  {64, 32, 4, 16.7f, 19.9f, 34.7f, 35.8f},  {64, 64, 2, 23.9f, 26.3f, 48.5f, 49.0f},
    {64, 128, 2, 28.6f, 36.2f, 67.0f, 70.0f}, {128, 256, 1, 73.0f, 88.0f, 153.0f, 160.0f}};

TileChoice w_tile_i4(int64_t group, int64_t m, int64_t n, int64_t k, int cus) {
  const TileCost& t = group == 32 ? kI4Tiles32[cheapest_tile(kI4Tiles32, m, n, k, cus)]
                                  : kI4Tiles[cheapest_tile(kI4Tiles, m, n, k, cus)];
  return {t.bm, t.bn, t.wk, kOneTile};
}

template <int KIND>
static int launch_kind(const WTileArgs& p, int splits, int cus, hipStream_t st) {
  // split K keeps the largest tile: its callers split products whose 128 x 256 tiles are few
  if constexpr (kind_group(KIND) == 32) {
    switch (p.part ? 4 : cheapest_tile(kI4Tiles32, p.M, p.N, p.K, cus)) {
      case 0: return launch_w_tile<KIND, 1, 1, 4, 3>(p, 1, st);
      case 1: return launch_w_tile<KIND, 2, 1, 4, 2>(p, 1, st);
      case 2: return launch_w_tile<KIND, 2, 2, 2, 3>(p, 1, st);
      case 3: return launch_w_tile<KIND, 2, 4, 2, 2>(p, 1, st);
      default: return launch_w_tile<KIND, 4, 8, 1, 2>(p, splits, st);
    }
  } else {
    switch (p.part ? 5 : cheapest_tile(kI4Tiles, p.M, p.N, p.K, cus)) {
      case 0: return launch_w_tile<KIND, 1, 1, 4, 3>(p, 1, st);
      case 1: return launch_w_tile<KIND, 1, 2, 4, 3>(p, 1, st);
      case 2: return launch_w_tile<KIND, 2, 2, 2, 3>(p, 1, st);
      case 3: return launch_w_tile<KIND, 2, 4, 2, 2>(p, 1, st);
      case 4: return launch_w_tile<KIND, 2, 4, 1, 3>(p, 1, st);
      default: return launch_w_tile<KIND, 4, 8, 1, 2>(p, splits, st);
    }
  }
}

int launch_gemm_w_tile_i4(const WTileArgs& p, int64_t block_size, int splits, int cus, hipStream_t st) {
  if (!p.scales) return launch_kind<kKindI4>(p, splits, cus, st);
  const bool wide = p.sdt == TGM_F32;
  if (wide || p.sdt == TGM_F16 || p.sdt == TGM_BF16) {
    switch (block_size) {
      case 32: return wide ? launch_kind<kKindI4 + 33>(p, splits, cus, st) : launch_kind<kKindI4 + 32>(p, splits, cus, st);
      case 64: return wide ? launch_kind<kKindI4 + 65>(p, splits, cus, st) : launch_kind<kKindI4 + 64>(p, splits, cus, st);
      case 128: return wide ? launch_kind<kKindI4 + 129>(p, splits, cus, st) : launch_kind<kKindI4 + 128>(p, splits, cus, st);
    }
  }
  TGM_UNSUPPORTED("tgm_gemm_w: int4 scales must be f16, bf16 or f32 per 32, 64 or 128 K-elements");
}

}  // namespace tgm
