"""Shapes at which the plans of the kernels for any mode sizes take each number
of tiles per wave: shared by the GPU tests of the results and the CPU test that
the shapes do reach them."""

# float64, shape, rank, mode, weights, tiles per wave.  Contracted inner modes
# shorter and longer than a lane's values, rank tiles 1 to 4, a slab past 64.
MTTKRP = [
    (False, (8, 62, 153, 9), 16, 2, False, 2), (False, (16513, 2), 5, 0, False, 2), (False, (42, 18, 105, 9), 20, 2, True, 2),
    (False, (20195, 2), 31, 0, False, 2), (False, (301, 13, 18, 9), 48, 2, True, 2), (False, (38, 56, 21, 9), 50, 2, True, 2),
    (False, (7, 179, 137, 10), 5, 2, False, 3), (False, (9, 231, 43, 3), 5, 2, False, 3),
    (False, (287, 475, 14), 20, 1, True, 3), (False, (175, 12, 37, 2), 31, 2, True, 3),
    (False, (419, 296, 11), 48, 1, True, 3), (False, (28, 84, 46, 2), 48, 2, False, 3),
    (False, (812, 34, 35), 64, 1, True, 3), (False, (81, 37, 51, 9), 5, 2, False, 4),
    (False, (129, 11, 117, 5), 16, 2, True, 4), (False, (39, 34, 107, 9), 20, 2, False, 4),
    (False, (135, 1206, 2), 20, 1, True, 4), (False, (24873, 601), 63, 0, False, 4),
    (False, (4, 70), 5, 1, False, 2), (False, (2, 65), 5, 1, False, 2),
    (False, (17, 29, 50, 143), 16, 3, False, 3), (False, (27, 310, 3, 156), 5, 3, False, 3),
    (True, (17985, 5), 16, 0, False, 2), (True, (24067, 2), 5, 0, False, 2), (True, (21233, 5), 20, 0, True, 2),
    (True, (12653, 7), 37, 0, False, 2), (True, (13847, 5), 50, 0, False, 2), (True, (752, 165, 5), 16, 1, True, 3),
    (True, (60, 24, 68, 2), 5, 2, True, 3), (True, (312, 141, 21), 20, 1, True, 3), (True, (56, 32, 33, 3), 20, 2, False, 3),
    (True, (20567, 7), 48, 0, True, 3), (True, (365, 401, 5), 16, 1, False, 4), (True, (64, 13, 152, 2), 16, 2, False, 4),
    (True, (4136, 485), 20, 0, True, 4), (True, (4, 39), 5, 1, True, 2), (True, (2, 35), 16, 1, False, 2),
    (True, (14, 251, 7, 79), 16, 3, False, 3), (False, (300, 41, 900), 100, 1, True, None),
    (True, (300, 41, 500), 90, 1, True, None),
]

# float64, shape, mode, J, tiles per wave, the waves of a block share a tile
MODE_DOT = [
    (False, (2100, 35, 250), 1, 16, 2, False), (False, (2100, 35, 251), 1, 31, 2, False), (False, (2101, 35, 250), 1, 33, 1, False),
    (False, (1100, 35, 130), 1, 16, 1, True), (False, (262_201, 19), 1, 16, 4, False), (False, (262_201, 35), 1, 33, 2, False),
    (False, (262_201, 19), 1, 64, 2, False), (True, (4101, 35, 125), 1, 16, 2, False), (True, (4101, 35, 125), 1, 64, 1, False),
    (True, (1100, 37, 67), 1, 17, 1, True), (True, (262_201, 19), 1, 16, 4, False), (True, (262_201, 35), 1, 64, 2, False),
]
