"""Sizes (M, N, K) that reach every tile of the matrix products on an MI355X, ragged in M and N.

The GPU tests check each product's values; the host test holds the sizes to what the entry points choose for 256
compute units, so that a changed choice cannot leave a kernel untested.  A tile is (rows, columns, groups of waves that
share its K steps, kernel), the kernel 0 for the one-tile kernels, 1 for a kernel of large tiles, 2 for a persistent one.
"""

import ctypes

from tinygrad_mi355x.runtime import library as L

CUS = 256


def _ask(name: str, *args) -> tuple[int, int, int, int]:
    tile = (ctypes.c_int64 * 4)()
    L.call(name, *args, CUS, tile)
    return tuple(tile)


def weight_tile(fmt, group, m, n, k):
    return _ask("tgm_gemm_w_tile", L.FORMAT_IDS[fmt], group, m, n, k)


def pair_tile(fa, fb, scaled, m, n, k):
    return _ask("tgm_gemm_mx_tile", L.FORMAT_IDS[fa], L.FORMAT_IDS[fb], int(scaled), m, n, k)


def dense_tile(m, n, k):
    return _ask("tgm_gemm_dense_tile", m, n, k)


# Packed weights: a single K step, and 9, 10 and 11 steps, of which four groups of waves leave one, two and three idle.
WEIGHT_SIZES = [(17, 33, 128), (40, 1000, 640), (17, 33, 1152), (20, 1000, 1280), (40, 1030, 1408), (129, 2050, 1152),
                (70, 4100, 384), (70, 4100, 1280), (130, 4100, 1152), (200, 6150, 640), (500, 6150, 384),
                (515, 6150, 1152), (1030, 6150, 256), (1030, 4104, 640)]
WEIGHT_PERSISTENT = [(1000, 8200, 1024)]
WEIGHT_TILES = {
    "fp4_e2m1": {(32, 32, 4, 0), (32, 64, 4, 0), (64, 64, 2, 0), (64, 128, 1, 0), (128, 128, 1, 0), (128, 256, 1, 0),
                 (128, 256, 1, 2)},
    "fp6": {(32, 32, 4, 0), (64, 64, 2, 0), (64, 128, 1, 0), (128, 128, 1, 0), (128, 256, 1, 0), (128, 256, 1, 2)},
    "int4": {(32, 32, 4, 0), (32, 64, 4, 0), (64, 64, 2, 0), (64, 128, 2, 0), (64, 128, 1, 0), (128, 256, 1, 0)},
    "int4 groups of 32": {(32, 32, 4, 0), (64, 32, 4, 0), (64, 64, 2, 0), (64, 128, 2, 0), (128, 256, 1, 0)},
}

# Pairs: one K step, partial last stages and partial last batches of scales.
PAIR_SIZES = [(20, 100, 128), (33, 1030, 640), (17, 33, 1152), (40, 1000, 1408), (130, 4100, 896), (129, 6150, 384),
              (250, 4110, 640), (515, 4110, 1152), (515, 12300, 1152), (515, 4110, 128), (700, 6150, 640),
              (1030, 6150, 896)]
PAIR_TILES = {
    0: {(32, 64, 4, 0), (64, 64, 2, 0), (64, 128, 2, 0), (128, 128, 2, 0), (256, 128, 1, 1)},
    1: {(32, 64, 4, 0), (64, 64, 2, 0), (64, 128, 2, 0), (128, 128, 2, 0), (128, 256, 1, 0), (256, 128, 1, 1)},
}
PAIR_TILES[2] = PAIR_TILES[1]  # by the number of 6-bit operands
# FP4 pairs with both scales and K a multiple of 256
FP4_PAIR_SIZES = [(17, 33, 768), (130, 4100, 512), (250, 4110, 768), (515, 4110, 1280), (1030, 4104, 768),
                  (700, 6150, 1280), (1030, 4104, 1024)]
FP4_PAIR_TILES = {(32, 64, 4, 0), (64, 64, 2, 0), (64, 128, 2, 0), (128, 128, 2, 0), (256, 256, 1, 1), (256, 256, 1, 2)}

# bf16 / f16: K steps of 64
DENSE_SIZES = [(17, 72, 64), (33, 1032, 192), (40, 1000, 832), (200, 3104, 832), (70, 8200, 320), (257, 4104, 704),
               (515, 4104, 448), (515, 8184, 64), (1030, 4104, 192), (1030, 7688, 320)]
DENSE_PERSISTENT = [(4104, 4096, 128)]
DENSE_TILES = {(32, 64, 4, 0), (64, 64, 2, 0), (64, 128, 2, 0), (128, 128, 1, 0), (128, 256, 1, 0), (256, 256, 1, 2)}
