"""The smaller tiles of the INT8 products (oz_gemm_tiles.hip): digits and Scheme I diagonals exact at the
sizes where each tile's rule begins and ends, with K steps that do not divide among the waves or stages.

The reference is the product in float64 (BLAS), which is exact: every sum is an integer below 2^53."""
import numpy as np
import pytest

from oztt_amd.device import crt_desc, hip, to_blocks

pytestmark = pytest.mark.gpu

MODULI = [255, 254, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193, 191, 181, 179, 173, 167, 163, 157, 151]


def planes(rng, S, R, K):
    X = rng.integers(-127, 128, (S, R, K), dtype=np.int8)
    X[:, 0, :] = 127  # the largest sums
    X[:, -1, :] = -127
    return X


# The tile that each size stands for is asked of the rule (256 compute units).
TILE256, TILE256X128, TILE128, TILE64, SPLIT4, SPLIT8 = range(6)


@pytest.mark.parametrize("tile,M,N,K,S", [
    (TILE64, 256, 256, 64, 1), (TILE64, 256, 256, 512, 16), (TILE64, 512, 256, 192, 16),
    (SPLIT8, 256, 256, 576, 16), (SPLIT8, 256, 256, 1088, 3),         # 64 x 64, K over 8 waves
    (SPLIT4, 512, 256, 576, 16),                                      # ... over 4 waves
    (TILE128, 512, 512, 64, 16), (TILE128, 768, 768, 128, 16), (TILE128, 512, 768, 576, 13),
    (TILE256X128, 1024, 1024, 448, 16), (TILE256X128, 1536, 1024, 64, 16), (TILE256X128, 256, 6656, 192, 16),
    (TILE256, 1280, 1280, 1536, 16), (TILE256, 768, 768, 1088, 24),   # tiles not a multiple of 8: ranges per XCD
])
def test_digits_in_small_tiles(dev, tile, M, N, K, S):
    assert hip().oz_rule_digit_tile(256, M, N, K, S) == tile
    rng = np.random.default_rng(M + 3 * N + K + S)
    A, Bt = planes(rng, S, M, K), planes(rng, S, N, K)
    desc = crt_desc(MODULI[:S], 54, 3)
    bA, bB, bD = dev.upload(to_blocks(A)), dev.upload(to_blocks(Bt)), dev.alloc(S * M * N)
    dev.fill_u32(bD, 0xA5A5A5A5, S * M * N // 4)
    dev.gemm_digits(bA, bB, bD, M, N, K, S, N, M * K, N * K, M * N, desc)
    got = dev.download(bD, np.uint8, S * M * N).reshape(S, M, N)
    for s, m in enumerate(MODULI[:S]):
        C = (A[s].astype(np.float64) @ Bt[s].astype(np.float64).T).astype(np.int64)
        want = (C % m) * desc.y[s] % m
        assert got[s].max() <= m
        np.testing.assert_array_equal(got[s] % m, want, err_msg=f"modulus {m}")
    for x in (bA, bB, bD):
        x.free()
    dev.bufs.clear()


DIAG256, ALL, DIAG128, DIAG64, SPLIT64, SPLIT32 = range(6)


@pytest.mark.parametrize("tile,M,N,K,p", [
    (SPLIT32, 256, 256, 64, 2), (SPLIT32, 256, 256, 192, 13),         # 32 x 32, K over 4 waves
    (DIAG64, 512, 512, 128, 8), (DIAG64, 512, 256, 64, 3),
    (SPLIT64, 512, 512, 192, 7), (SPLIT64, 512, 256, 640, 10),        # 64 x 64, K over 8 waves
    (ALL, 768, 1024, 512, 5), (ALL, 768, 768, 576, 6), (ALL, 1024, 768, 576, 7),  # odd and even steps
    (ALL, 768, 768, 512, 8), (ALL, 768, 768, 576, 9), (ALL, 2048, 1024, 2048, 8),
    (DIAG128, 768, 768, 448, 8), (DIAG128, 768, 768, 576, 10), (DIAG128, 2048, 1024, 128, 4), (DIAG128, 1536, 2048, 384, 5),
    (DIAG256, 1280, 1280, 128, 11), (DIAG256, 1536, 1536, 192, 8),
])
def test_diagonals_in_small_tiles(dev, tile, M, N, K, p):
    assert hip().oz_rule_diag_tile(256, M, N, K, p) == tile
    dmax = 127 if p * K * 127 * 127 < 2**31 else 32
    rng = np.random.default_rng(M + 3 * N + K + p)
    A, Bt = (np.clip(planes(rng, p, R, K), -dmax, dmax) for R in (M, N))
    bA, bB, bP = dev.upload(to_blocks(A)), dev.upload(to_blocks(Bt)), dev.alloc(4 * p * M * N)
    dev.fill_u32(bP, 0xA5A5A5A5, p * M * N)
    dev.oz1_gemm_diag(bA, bB, bP, M, N, K, p, N, M * K, N * K, M * N, dmax)
    got = dev.download(bP, np.int32, p * M * N).reshape(p, M, N)
    Af, Bf = A.astype(np.float32), np.ascontiguousarray(Bt.astype(np.float32).transpose(0, 2, 1))
    for d in range(p):
        want = np.zeros((M, N))
        for i in range(d + 1):
            for k in range(0, K, 512):  # float32 sums of 512 products stay below 2^24
                want += Af[i][:, k:k + 512] @ Bf[d - i][k:k + 512]
        np.testing.assert_array_equal(got[d], want, err_msg=f"diagonal {d}")
    for x in (bA, bB, bP):
        x.free()
    dev.bufs.clear()
