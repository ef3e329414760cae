"""Sizes that run each W4A16, scaled fp8 and plain-product tile (tilebench_amd/csrc/small_plan.h), shared by
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
#: (tile, 16-byte weight loads) -> (tokens, experts, top k, K, columns, group) of the gate/up
#: (columns I: 16-byte loads where I % 32 == 0) and down products (columns H, likewise):
#: tokens routed nowhere, an expert without rows or with several row tiles, ragged last column tiles
GATE_UP_TILES = {
    ("32x128", True): (33, 5, 3, 320, 96, 64), ("32x128", False): (33, 5, 3, 320, 72, 64),
    ("32x256", True): (70, 70, 2, 192, 704, 64), ("32x256", False): (70, 70, 2, 128, 712, 128),
    ("64x256", True): (500, 32, 4, 128, 704, 64), ("64x256", False): (500, 32, 4, 192, 712, 64),
    ("256", True): (1500, 16, 4, 128, 704, 64), ("256", False): (1500, 16, 4, 64, 712, 64),
}
DOWN_TILES = {
    ("32x128", True): (33, 5, 3, 192, 320, 64), ("32x128", False): (33, 5, 3, 64, 328, 64),
    ("32x256", True): (24, 64, 8, 192, 1408, 64), ("32x256", False): (70, 70, 2, 128, 1416, 128),
    ("64x256", True): (500, 32, 4, 192, 1408, 64), ("64x256", False): (500, 32, 4, 64, 1416, 64),
    ("256", True): (1500, 16, 4, 128, 1408, 64), ("256", False): (1500, 16, 4, 64, 1416, 64),
}
EXPERT_TILE_IDS = {"256": 0, "32x128": 1, "32x256": 2, "64x256": 3}

#: tile -> (M, K, N, group) of the dense product: ragged rows and columns, K of
#: fewer steps than K groups, N % 32 != 0
DENSE_TILES = {
    "64x64": [(17, 64, 8, 64), (33, 320, 392, 64), (64, 704, 1000, 64), (48, 2048, 4096, 128)],
    # up to 64 rows too where N alone fills the device
    "64x128": [(65, 64, 264, 64), (129, 448, 1096, 64), (500, 192, 4096, 64), (64, 64, 32768, 64)],
    "64x256": [(300, 192, 22040, 64), (1000, 128, 4096, 64), (40, 64, 65536, 64)],
    "128x256": [(768, 320, 8944, 64), (2047, 64, 4096, 64)],
    # half a round and more of 256 x 256 tiles: two rounds and a bit of a smaller tile take 20 - 28 % longer
    "256": [(1024, 192, 11008, 64), (691, 192, 11896, 64), (729, 64, 12288, 64), (1725, 64, 5480, 64),
            (2204, 64, 4096, 64), (4086, 64, 2216, 64)],
}
DENSE_TILE_IDS = {"256": 0, "64x64": 1, "64x128": 2, "64x256": 3, "128x256": 4}

#: tile -> (M, N, K) of the scaled fp8 products (both scalings): ragged rows and
#: columns, one K step, fewer K steps than wavefronts or ring stages, odd step
#: counts, one and several tiles per CU
FP8_TILES = {
    "32x32": [(1, 8, 128), (31, 2112, 1408), (16, 8184, 896)],
    "64x64": [(65, 4000, 640), (126, 4104, 128), (200, 2112, 1152)],
    "64x128": [(126, 8200, 128), (300, 5000, 384)],
    "128x128": [(512, 4104, 640), (600, 8200, 1024)],
    "256": [(1024, 8200, 1152)],
}
FP8_TILE_IDS = {"256": 0, "32x32": 1, "64x64": 2, "64x128": 3, "128x128": 4}

#: tile -> (M, N, bytes of K per row) of the plain products: ragged rows and
#: columns, one K step, odd step counts, one and several tiles per CU
NT_TILES = {
    "64x64": [(1, 8, 128), (65, 1000, 640), (100, 4104, 1152)],
    "64x128": [(513, 2056, 640), (300, 5000, 384)],
    # the last two: just over one tile per CU on many steps, and half a round of 256 x 256 tiles on few
    "128x128": [(1000, 2104, 1152), (1100, 5000, 640), (3380, 1192, 3840), (2779, 3616, 256)],
    "256": [(4096, 4104, 1152)],
}
NT_TILE_IDS = {"256": 0, "64x64": 1, "64x128": 2, "128x128": 3}

#: (columns of a slab, K splits on 256 CUs) -> (N, K) of the W4A16 decode: one
#: column, ragged and odd numbers of slabs, K of fewer units than wavefronts, unequal
#: shares of the units, half-filled 16-column lanes at 256 columns
DECODE_PLANS = {
    (128, 1): [(8, 64), (136, 192), (2048, 1024), (264, 128)],
    (128, 3): [(9000, 3072), (10112, 3200)],
    (128, 4): [(1408, 4096), (4096, 4096), (5000, 3072)],
    (128, 8): [(4096, 11008)],
    (256, 1): [(32776, 1024)],
    (256, 5): [(12288, 4096), (12296, 4096)],
    (256, 7): [(8944, 6080)],
}
