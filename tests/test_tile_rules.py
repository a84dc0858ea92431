"""The rules by which a launch of INT8 products takes its tiles and their order (oz_gemm_tiles.hip, oz_gemm.hip), and the
scale cuts strips of columns (oz_scale.hip), at sizes on either side of their lines, on 256 compute units. Every choice was measured against the others at the size
given. CPU only: the library's own rules are asked."""
import pytest

from oztt_amd.device import hip

CUS = 256


@pytest.mark.parametrize("M,N,K,batch,ranges", [
    (1024, 1024, 1024, 16, 1),    # one tile per CU: whole products per XCD
    (2048, 2048, 1536, 4, 1),
    (1280, 1280, 2048, 16, 1),    # 8 does not divide a product's tiles
    (1536, 1536, 2048, 14, 1), (1536, 1536, 2048, 20, 1), (2560, 2560, 1536, 10, 1), (3840, 3840, 4096, 17, 1),
    (2304, 2304, 8192, 15, 0),    # ... but eight products' operands pass the Infinity Cache
    (3328, 3328, 8192, 12, 0), (3328, 3328, 8192, 5, 1),
    (2304, 2304, 8192, 16, 1),    # whole products per XCD
    (2048, 2048, 2048, 15, 0), (8192, 8192, 8192, 15, 0), (2048, 1536, 2048, 10, 0),
])
def test_order_of_the_large_tiles(M, N, K, batch, ranges):
    assert hip().oz_rule_tile_ranges(CUS, M, N, K, batch) == ranges


TILE256, TILE256X128, TILE128, TILE64, SPLIT4, SPLIT8 = range(6)


@pytest.mark.parametrize("M,N,K,S,tile", [
    (256, 256, 512, 16, TILE64), (256, 256, 576, 16, SPLIT8), (512, 256, 576, 16, SPLIT4), (512, 512, 64, 16, TILE128),
    (512, 512, 8192, 16, TILE128), (768, 768, 2048, 16, TILE128), (768, 768, 2112, 16, TILE256),
    (1024, 768, 1024, 16, TILE128), (1024, 1024, 448, 16, TILE256X128), (1024, 1024, 512, 16, TILE256),
    (2048, 2048, 1024, 16, TILE256X128), (2048, 2048, 1088, 16, TILE256),
    (1536, 1024, 8192, 16, TILE256X128),                                # 384 large tiles: three quarters of two rounds
    (1280, 1024, 2048, 20, TILE256), (1280, 1280, 8192, 16, TILE256), (1792, 1792, 4096, 8, TILE256),  # a little more
    (2304, 2304, 3072, 5, TILE256), (2304, 2304, 1024, 5, TILE256X128),
])
def test_tiles_of_the_digits(M, N, K, S, tile):
    assert hip().oz_rule_digit_tile(CUS, M, N, K, S) == tile


DIAG256, ALL, DIAG128, DIAG64, SPLIT64, SPLIT32 = range(6)


@pytest.mark.parametrize("M,N,K,p,tile", [
    (256, 256, 512, 8, SPLIT32), (512, 512, 128, 8, DIAG64), (512, 512, 192, 8, SPLIT64),
    (1024, 1024, 448, 8, DIAG128), (1024, 1024, 512, 8, ALL), (2048, 1024, 1984, 8, DIAG128), (2048, 1024, 2048, 8, ALL),
    (2048, 2048, 192, 8, DIAG128), (2048, 2048, 448, 8, DIAG256), (4096, 4096, 384, 8, DIAG128),
    # more slices than the all-diagonals kernel has, or fewer: by the share of their time that large tiles fill
    (1024, 768, 8192, 10, DIAG128), (2048, 1024, 1024, 10, DIAG128), (2048, 1024, 8192, 4, DIAG128),
    (2048, 1024, 512, 13, DIAG256), (2048, 1024, 8192, 11, DIAG256), (256, 8192, 8192, 13, DIAG256),
    (2048, 1024, 4096, 16, DIAG256), (2048, 1024, 128, 12, DIAG128), (256, 8192, 256, 16, DIAG128),
    (1280, 1280, 128, 11, DIAG256), (1280, 1280, 1024, 11, DIAG128), (1280, 1280, 8192, 11, DIAG256),
    (1280, 1280, 4096, 13, DIAG256), (1536, 1024, 8192, 16, DIAG256), (1536, 1024, 8192, 10, DIAG128),
    (1536, 1536, 192, 8, DIAG256), (2048, 1536, 256, 7, DIAG256), (2304, 2304, 384, 5, DIAG256),
    (2048, 2048, 256, 4, DIAG128), (2816, 2816, 384, 2, DIAG128), (3072, 3072, 384, 3, DIAG256),
    (3584, 3584, 384, 12, DIAG256), (4096, 4096, 384, 16, DIAG256), (2048, 2048, 384, 10, DIAG128),
])
def test_tiles_of_the_diagonals(M, N, K, p, tile):
    assert hip().oz_rule_diag_tile(CUS, M, N, K, p) == tile


@pytest.mark.parametrize("M,N,K,cut", [
    (64, 2048, 1024, False), (256, 256, 1025, True), (64, 2048, 1100, True), (2048, 2048, 1025, False), (16, 2500, 1200, True),
    (2048, 2500, 1200, False), (512, 3000, 1025, False), (16, 4096, 2048, False), (16, 4096, 4096, True),
    (2048, 2048, 4096, True), (4096, 4096, 4096, False), (8192, 64, 8192, True), (8192, 1024, 8192, False),
    (4096, 1024, 4096, True), (2048, 3000, 8192, True), (4096, 3000, 3072, False), (256, 256, 32768, True),
    (64, 4097, 32768, False),
])
def test_strips_that_the_scale_cuts(M, N, K, cut):
    assert (hip().oz_rule_strip_chunks(CUS, M, N, K) > 1) == cut
