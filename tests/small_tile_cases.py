"""Sizes that run each W4A16 tile (tilebench_amd/csrc/small_plan.h), shared by
the CPU check of the rule and the GPU parity tests."""

#: tile -> (rows per expert, N of the product, K, group): rows on both sides of
#: the tile's edges, an empty expert, last column tiles of 8, 72 and 136 columns
#: (N % 32 != 0 takes the 4-byte weight loads), 1, 3 and 5 K steps
EXPERT_TILES = {
    "32x128": [([1, 0, 31, 32, 33, 2], 264, 320, 64), ([3, 5, 1], 128, 64, 64), ([40, 7, 0, 9], 200, 192, 192)],
    "32x256": [([33, 1, 0, 32, 31, 64, 5, 17] * 8, 1408, 192, 64), ([2] * 70, 1096, 128, 128)],
    "64x256": [([63, 64, 65, 1, 0, 129, 128, 40] * 8, 1408, 192, 64), ([100] * 33, 2056, 320, 64)],
    "256": [([600, 511, 700, 0, 512, 513, 900, 255] * 8, 1408, 128, 64)],
}
EXPERT_TILE_IDS = {"256": 0, "32x128": 1, "32x256": 2, "64x256": 3}
