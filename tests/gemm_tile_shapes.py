"""Shapes at the edges of the tile GEMM's configurations, shared by the test of
the products (test_gpu_gemm_tile.py) and the test that each runs the named
configuration (test_dispatch.py): rows, columns (SwiGLU: act columns), K, the
16-row fragments per wave (FM, FN: tiles of 32 FM rows x 32 FN weight rows) and
the most tiles that one of at most 256 workgroups takes in turn."""

FP8 = [
    (257, 16392, 1024, (8, 8), 1),    # one row and 8 columns in the last tiles
    (513, 40712, 1024, (8, 8), 2),    # 480 tiles: the ring runs on into the second
    (1281, 40712, 1024, (8, 8), 4),   # 960 tiles
    (513, 9864, 4096, (8, 4), 1),
    (1281, 10760, 3072, (8, 4), 2),
    (17, 38216, 2048, (4, 6), 1),
    (513, 26120, 2048, (4, 6), 3),    # 685 tiles
    (129, 12808, 1536, (4, 4), 1),
    (257, 16392, 1536, (4, 4), 2),    # 387 tiles
    (65, 12808, 1024, (4, 2), 1),     # two K groups from here on
    (257, 4936, 1024, (4, 2), 1),
    (17, 25480, 2560, (2, 4), 1),
    (17, 51080, 2560, (2, 4), 2),     # 400 tiles
    (65, 8200, 1024, (2, 3), 1),
    (17, 19112, 1024, (2, 3), 1),
    (65, 4104, 1024, (2, 2), 1),
    (17, 8200, 1024, (2, 2), 1),
    (33, 40, 1536, (2, 1), 1),
    (17, 8, 1024, (2, 1), 1),
    (16, 6152, 2048, (2, 1), 1),      # 16 rows, more skinny workgroups than CUs
    (2053, 520, 1024, (2, 3), 1),     # tiles numbered along N from here on
    (2820, 1032, 1536, (4, 4), 1),
    (6700, 4104, 1024, (8, 8), 2),    # 459 tiles
]
BF16 = [
    (257, 16392, 512, (8, 8), 1),
    (257, 50950, 512, (8, 8), 2),     # 400 tiles; odd groups of 8 columns, even pitch
    (1281, 25606, 512, (8, 8), 3),    # 606 tiles
    (513, 9864, 768, (8, 4), 1),
    (1281, 10760, 512, (8, 4), 2),    # 510 tiles
    (17, 38216, 512, (4, 6), 1),
    (257, 38214, 512, (4, 6), 3),     # 600 tiles
    (129, 12806, 512, (4, 4), 1),     # two K groups from here on
    (257, 16392, 1536, (4, 4), 2),    # 387 tiles
    (700, 3080, 2048, (4, 3), 1),
    (513, 13064, 4096, (4, 3), 3),    # 685 tiles
    (65, 8198, 512, (2, 4), 1),
    (17, 51080, 512, (2, 4), 2),      # 400 tiles
    (193, 4104, 2048, (2, 3), 1),
    (33, 136, 512, (2, 2), 1),
    (17, 38, 512, (2, 2), 1),
    (33, 42, 1024, (1, 2), 1),
    (17, 40, 2048, (1, 1), 1),        # four K groups
    (9, 8200, 512, (2, 2), 1),        # 9 rows, more skinny workgroups than CUs
    (2053, 520, 512, (2, 4), 1),      # tiles numbered along N from here on
    (2307, 2054, 512, (4, 6), 1),
    (6700, 3078, 512, (8, 4), 3),     # 675 tiles
]
SWIGLU = [
    (17, 16392, 768, (8, 8), 1),
    (513, 20360, 768, (8, 8), 2),     # 480 tiles
    (1281, 20360, 1536, (8, 8), 4),   # 960 tiles
    (257, 5448, 4096, (8, 4), 1),
    (1281, 5384, 3072, (8, 4), 2),    # 510 tiles
    (17, 136, 512, (4, 4), 1),
    (257, 25544, 2048, (4, 4), 5),    # 1200 tiles
    (65, 4104, 1024, (2, 4), 1),
    (17, 8200, 1024, (2, 4), 1),
    (17, 40, 1024, (2, 2), 1),
    (300, 520, 1536, (2, 2), 1),
    (16, 8264, 3584, (2, 4), 1),      # 16 rows, more skinny workgroups than CUs
    (2820, 520, 512, (4, 4), 1),      # tiles numbered along N from here on
    (6700, 2056, 1024, (8, 8), 2),    # 459 tiles
]
# K too short for a tile, or fewer rows than it takes: the general and the skinny kernels.
FP8_OTHER = [(17, 40, 256), (17, 136, 512), (2049, 2600, 256), (700, 8200, 512), (129, 8200, 1024),
             (16, 12808, 512)]
BF16_OTHER = [(17, 38, 128), (129, 136, 256), (700, 8200, 256), (2500, 2600, 128)]
SWIGLU_OTHER = [(17, 40, 256), (129, 8200, 512), (2049, 1288, 256), (16, 8200, 512)]


def tiles(m, n, fragments, glu=False):
    """Tiles of a shape: 32 FM rows x 32 FN columns (SwiGLU: 16 FN)."""
    return -(-m // (32 * fragments[0])) * -(-n // ((16 if glu else 32) * fragments[1]))
