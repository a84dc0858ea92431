"""oz_scale_pair_f64 where B's columns are few and long (K > 1024): a strip of columns is cut into runs of 512
rows and more, whose maxima meet in the handle. Against the oracle's scale, with the special values in
different runs; twice, since the last run clears what the strip used."""
import numpy as np
import pytest

from oztt_amd.device import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(1, 1025), (31, 1536), (33, 1537), (32, 2050), (65, 9001), (4096, 1100), (12, 33000), (4077, 3100),
                                 (2499, 1300)])
def test_chunked_columns_match_oracle(dev, oracle, N, K):
    M, lda, ldb, shift = 9, K + 2, N + 3, 16
    assert (hip().oz_rule_strip_chunks(256, M, N, K) > 1) == ((N, K) != (4096, 1100))  # (whole strips there)
    rng = np.random.default_rng(N + K)
    A = np.full((M, lda), 1e300)
    A[:, :K] = rng.uniform(-1, 1, (M, K))
    B = np.full((K, ldb), 1e300)
    B[:, :N] = rng.uniform(-1, 1, (K, N)) * np.exp2(rng.integers(-30, 30, (1, N)))
    special = [(0.0, 0), (2.0 ** -130, K - 1), (float.fromhex("0x1.ff8p127"), 511), (np.nan, 512), (-np.inf, K // 2),
               (float.fromhex("0x1.fep127"), 1023), (2.0 ** -126, 1024), (float.fromhex("0x1.fe00000000001p127"), K - 2)]
    bA, dA, dB, fl = dev.upload(A), dev.alloc(4 * M), dev.alloc(4 * N), dev.alloc(8)
    for first in (0, N):  # with special columns, then without
        X = B.copy()
        for i, (v, k) in enumerate(special):
            if first + i < N:
                X[:, first + i] = 0.0 if abs(v) < 1e-30 else X[:, first + i]
                X[k, first + i] = v
        bB = dev.upload(X)
        dev.fill_u32(fl, 0, 2)
        dev.scale_pair(bA, M, K, lda, bB, N, ldb, 1, shift, dA, dB, fl)
        got, flags = dev.download(dB, np.int32, N), dev.download(fl, np.uint32, 2)
        gA = dev.download(dA, np.int32, M)
        bB.free()
        want, wf = oracle.scale(np.ascontiguousarray(X[:, :N]), K, N, 1, 1, shift)
        wA, wfA = oracle.scale(np.ascontiguousarray(A[:, :K]), M, K, 0, 1, shift)
        np.testing.assert_array_equal(got, want)
        np.testing.assert_array_equal(gA, wA)
        assert list(flags) == [wfA, wf]
    for x in (bA, dA, dB, fl):
        x.free()
    dev.bufs.clear()
