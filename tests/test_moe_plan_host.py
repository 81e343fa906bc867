"""The rule that takes experts of 256 to 767 rows to the 256-row tiles."""
from sglang_amd import kernels as K


def test_experts_of_middling_size():
    for pairs, experts, up, down, rows in ((2 * 3000, 8, 14336, 4096, 256), (2 * 3000, 8, 7168, 4096, 256), (6 * 6000, 64, 1408, 2048, 256),
                                           (2 * 2300, 8, 14336, 4096, 256), (2 * 6000, 16, 2048, 2048, 256),
                                           (2 * 2000, 8, 7168, 4096, 128), (2 * 1000, 8, 14336, 4096, 128), (2 * 4000, 16, 2048, 2048, 128),
                                           (2 * 1622, 8, 14336, 4096, 128), (2 * 2048, 8, 14336, 4096, 128),
                                           (2 * 1020, 8, 14336, 4096, 128)):
        assert K.moe_tile_plan(pairs, experts, up, down) == (rows,) * 3, (pairs, experts, up, down)


def test_experts_that_half_tiles_pay_for():
    for pairs, experts, up, down, rows in ((2 * 1000, 8, 14336, 4096, 256), (2 * 1622, 8, 14336, 4096, 256), (2 * 2048, 8, 14336, 4096, 256),
                                           (2 * 3000, 8, 14336, 4096, 256), (32 * 260, 32, 7168, 4096, 256), (64 * 350, 64, 1408, 2048, 256),
                                           (2 * 950, 8, 14336, 4096, 128), (2 * 1600, 8, 7168, 4096, 128), (16 * 500, 16, 2048, 2048, 128),
                                           (64 * 200, 64, 4096, 2048, 128)):
        assert K.moe_tiles(pairs, experts, up, down) == (rows,) * 3, (pairs, experts, up, down)


def test_experts_that_even_tiles_pay_for():
    for pairs, experts, up, down, rows in ((64 * 140, 64, 1408, 2048, 256), (64 * 139, 64, 1408, 2048, 128), (8 * 140, 8, 14336, 4096, 256),
                                           (8 * 100, 8, 14336, 4096, 128), (32 * 230, 32, 2048, 2048, 128), (16 * 300, 16, 2048, 2048, 256),
                                           (16 * 299, 16, 2048, 2048, 128), (4 * 600, 4, 1024, 1024, 128), (8 * 1024, 8, 14336, 4096, 256)):
        assert K.moe_rows(pairs, experts, up, down) == (rows,) * 3, (pairs, experts, up, down)


def test_where_the_row_tiles_begin():
    for pairs, experts, up, tiled in ((8 * 56, 8, 14336, True), (8 * 55, 8, 14336, False), (4 * 95, 4, 1024, False), (4 * 96, 4, 1024, True),
                                      (8 * 56, 8, 2048, True), (8 * 1000, 8, 64, True)):
        assert K._row_tiled(pairs, experts, up) == tiled, (pairs, experts, up)
