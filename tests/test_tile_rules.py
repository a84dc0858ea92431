"""The rules by which a launch of INT8 products takes its tiles and their order (oz_gemm_tiles.hip, oz_gemm.hip), at
sizes on either side of their lines, on 256 compute units. Every choice was measured against the others at the size
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
